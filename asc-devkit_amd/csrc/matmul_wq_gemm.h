// The half GEMM on quantised weights (matmul_wq_gemm.hip), shared by W8A16 and W4A16.
#pragma once
#include "ascq_common.h"

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
    uint32_t tiles_m, tiles_n, full;  // (set by the launch)
    WqMasks mk;
};

// A lane addresses its row of a tile's 128 or 256 by 32 bits: longer rows stay with the passes over the weights.
constexpr uint32_t kWqMaxK = 1u << 23;
int launch_wq_gemm(const WqParams& p, bool int4, bool has_offset, hipStream_t st);

}  // namespace ascq
