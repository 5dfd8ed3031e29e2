// The two tile kernels of half x quantised weights (matmul_wq_gemm.hip, matmul_wq_rows.hip), shared by W8A16 and W4A16.
#pragma once
#include "ascq_common.h"
#include "ascq_device.h"

namespace ascq {

struct WqMasks {
    uint32_t even, odd, exp_even, exp_odd;
};

struct WqParams {
    const uint16_t* x;       // [m, k] halves, 16-byte aligned
    const uint8_t* w;        // int8 [n, k] (k % 64 == 0) or packed int4 (k % 128 == 0), 16-byte aligned
    const uint16_t* scale;   // int8: [n] halves, or nullptr for scale_bits / offset_bits; int4: [k / group_size, n]
    const uint16_t* offset;  // same (only read with an offset)
    void* y;                 // [m, n] halves or floats
    uint32_t m, n, k;
    uint32_t out_f32;
    uint32_t scale_bits, offset_bits;
    uint32_t gs_shift;       // int4: log2(group_size / 32)
    uint32_t tiles_m, tiles_n, full, wide_store;  // (set by the launch)
    WqMasks mk;
};

// ---- weights to halves, shared by the two kernels
__device__ __forceinline__ f16x2 as_h2(uint32_t b) { return __builtin_bit_cast(f16x2, b); }
__device__ __forceinline__ uint32_t as_u32(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f16x2 both(float v) { return f16x2{static_cast<half_t>(v), static_cast<half_t>(v)}; }

// two weights as exact halves -> with the operators' roundings: one for the offset, one for the scale
template <bool kOff>
__device__ __forceinline__ uint32_t finish(f16x2 w, f16x2 sc, f16x2 of)
{
    if constexpr (kOff) {
        w = w + of;
    }
    return as_u32(sc * w);
}

// pair c (of 2) of 4 int8: 0x6400 | (w + 128) is the half 1152 + w
template <bool kOff>
__device__ __forceinline__ uint32_t pair_of_i8(uint32_t d, int c, f16x2 sc, f16x2 of)
{
    const uint32_t flipped = d ^ 0x80808080u;  // w + 128 as an unsigned byte
    return finish<kOff>(as_h2(__builtin_amdgcn_perm(0x64646464u, flipped, c ? 0x04030402u : 0x04010400u)) - both(1152.0f), sc, of);
}

// pair c (of 4) of a dword of packed int4 (u = w + 8, k offsets 0 .. 7 in nibbles 0 4 1 5 2 6 3 7): 0x6400 | u is the
// half 1024 + u, 0x5400 | 16 u the half 64 + u
template <bool kOff>
__device__ __forceinline__ uint32_t pair_of_i4(uint32_t q, int c, f16x2 sc, f16x2 of, const WqMasks& mk)
{
    const uint32_t src = c & 2 ? q >> 8 : q;
    return c & 1 ? finish<kOff>(as_h2((src & mk.odd) | mk.exp_odd) - both(72.0f), sc, of)
                 : finish<kOff>(as_h2((src & mk.even) | mk.exp_even) - both(1032.0f), sc, of);
}

// Where piece q of a line of 128 bytes lies: at q ^ wq_swizzle(line).  16 neighbouring lines meet all 64 banks in a 16-byte
// read of one piece, and four neighbouring lines all 32 banks that a write sees at a time in two pieces four apart.
__device__ __forceinline__ uint32_t wq_swizzle(uint32_t line) { return ((line >> 1) & 7u) ^ ((line & 1u) << 1); }

// A lane addresses its row of a tile's 128 or 256 by 32 bits: longer rows stay with the passes over the weights.
constexpr uint32_t kWqMaxK = 1u << 23;
int launch_wq_gemm(const WqParams& p, bool int4, bool has_offset, hipStream_t st);
// us that launch_wq_gemm is expected to take
double wq_gemm_estimate(uint32_t m, uint32_t n, uint32_t k);

// Whole-k tiles of 16 to 64 rows and columns (matmul_wq_rows.hip): runs the call and returns true where they are expected to
// beat `other_us`, what the caller would do instead.  sum: int4 in group-sum form (group_size a multiple of 128).
bool wq_rows_ahead(const WqParams& p, bool int4, bool sum, bool has_offset, double other_us, hipStream_t st);
// us that the best of those tiles is expected to take
double wq_rows_estimate(uint32_t m, uint32_t n, uint32_t k, bool int4);

// us that a call on packed int4 (per weight) or [n, k] int8 weights is expected to take with 5 rows and more: for callers that
// would have to bring their weights into that form first
double w4a16_packed_estimate(uint32_t m, uint32_t n, uint32_t k);
double w8a16_nk_estimate(uint32_t m, uint32_t n, uint32_t k);

}  // namespace ascq
