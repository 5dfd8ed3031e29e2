// Half x quantised weights where the tiles of matmul_wq_gemm.hip would leave most of the chip idle (few rows or few columns), and the
// group-sum form of int4 weights with any number of rows.
//
// A workgroup of 8 wavefronts owns 16 to 64 rows by 16 to 64 columns over all of k: small tiles give every compute unit work, and k is
// split inside the workgroup, a contiguous run per wavefront, so that no partial sum leaves the compute unit.  A wavefront works alone:
// it fetches its part of x into LDS of its own (8 KiB per stage, two stages, no barrier, counted waits), its weights into registers
// (a lane's 16 k of a column are two operands of v_mfma_f32_16x16x32_f16), and the de-quantised weights never see the LDS.  What is read
// of a stage is in registers before the first product, so its place takes the loads of the stage after next at once: every load
// has one to two stages to arrive.  The eight partial tiles meet in LDS at the end, added in wavefront order.
//
// What bounds it is x on its way from L2 into the LDS, 64 KiB per stage of 64 x 64 products of 512 k (0.8 of 1.1 us at the 80 GB/s and
// compute unit that such loads reach), then the vector ALU's de-quantisation (17 operations per 8 weights, 0.5 us).  From passes over the
// weights per 16 rows, and 128 x 128 tiles, in us: int4 37 x 12288 x 2816 77 -> 16, 125 x 11264 x 3488 109 -> 23; int8 63 x 10880 x 1760
// 90 -> 17, 288 x 12928 x 1488 112 -> 32; group sums 37 x 4224 x 1408 17 -> 7, 1199 x 5120 x 5376 1067 -> 105.  Also built: tiles of 64 x 128 (128
// accumulators; 512 x 8192 x 28672 312 us, 64 x 64 357, the 256 x 256 tiles 203: with the chip full the traffic decides).
#include <type_traits>

#include "ascq_common.h"
#include "ascq_device.h"
#include "matmul_wq_gemm.h"

namespace ascq {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kWaves = 8;
constexpr uint32_t kStageBytes = 8192;  // of x per wavefront and stage
constexpr int kALoads = kStageBytes / 1024;

enum WqKind { kInt4Weight, kInt4Sum, kInt8Weight };

// Place of element (row, col) of a BM x BN tile of partial sums: the rows of a wavefront's four lane groups, four apart, lie in
// different banks.
template <int BN>
__device__ __forceinline__ uint32_t sum_place(uint32_t row, uint32_t col)
{
    return (row * BN + col) ^ (((row >> 2) & 3u) << 4);
}

// The loads of an even (0) or odd (1) stage.
template <int BM, int BN, int kKind, bool kOff>
struct StageLoads {
    // Whether a sub-step fetches parameters: with int8 none does; in the sum form those at the end of 128 k (loads that nobody uses the
    // compiler leaves out, and a count that includes them would not hold a wait back).
    static constexpr bool params(int parity, int s) { return kKind == kInt4Weight || (kKind == kInt4Sum && ((parity * (64 / BM) + s) & 1) != 0); }
    static constexpr int count(int parity)
    {
        int n = kALoads + 64 / BM * (BN / 16);
        for (int s = 0; s < 64 / BM; ++s) n += params(parity, s) ? BN / 16 * (kOff ? 2 : 1) : 0;
        return n;
    }
};

template <int BM, int BN, int kKind, bool kOff>
__global__ __launch_bounds__(kWaves * 64, 2) void wq_rows_kernel(WqParams p)
{
    constexpr bool kInt4 = kKind != kInt8Weight, kSum = kKind == kInt4Sum;
    constexpr int NI = BM / 16, NJ = BN / 16, SUB = 64 / BM;  // a stage: SUB times BM rows x 64 k
    constexpr int kParams = kInt4 ? SUB * NJ : 1;
    using Loads = StageLoads<BM, BN, kKind, kOff>;
    constexpr uint32_t kUnit = kInt4 ? 2u : 1u;               // a wavefront's share of k is a multiple of this many 64 k
    static_assert(NI * 16 == BM && NJ * 16 == BN && SUB * BM == 64, "tile shape");
    __shared__ __attribute__((aligned(1024))) char A0[kWaves * kStageBytes], A1[kWaves * kStageBytes];

    const uint32_t t = xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n);
    if (t == 0xFFFFFFFFu) {
        return;  // whole workgroup (the launch is rounded up to a multiple of 8)
    }
    uint32_t tm, tn;
    band_order(t, p.tiles_m, p.tiles_n, tm, tn);
    const uint32_t row0 = tm * BM, n0 = tn * BN;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, lc = lane & 15u, lq = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- this wavefront's k: 64 sub0 .. 64 sub_end - 1
    const uint32_t subs = p.k / 64u, units = subs / kUnit;
    const uint32_t sub0 = wave * units / kWaves * kUnit, sub_end = (wave + 1u) * units / kWaves * kUnit;
    const uint32_t stages = (sub_end - sub0 + SUB - 1u) / SUB;

    // ---- x: a stage is SUB * BM lines of 64 halves (sub-step major), lane l of load u owns 16-byte place u * 64 + l.  Rows past
    // the end lie outside the buffer: zeros, without a trip to memory
    constexpr int kRowLoads = BM / 8;                         // loads that cover the rows of a sub-step
    const uint32_t row_bytes = p.k * 2u;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.x) + static_cast<size_t>(row0) * p.k, 0, static_cast<int>((p.m - row0 < BM ? p.m - row0 : BM) * row_bytes), 0x00020000);
    uint32_t aoff[kRowLoads];
#pragma unroll
    for (int u = 0; u < kRowLoads; ++u) {
        const uint32_t r = u * 8u + (lane >> 3);
        aoff[u] = r * row_bytes + (((lane & 7u) ^ wq_swizzle(r)) << 4);
    }
    auto load_x = [&](char* S, uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            const uint32_t at = (sub0 + stage * SUB + s) * 128u;  // (past the end: whatever lies there, nobody reads it)
#pragma unroll
            for (int u = 0; u < kRowLoads; ++u) {
                const uint32_t off = aoff[u];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr_t)(S + wave * kStageBytes + (s * kRowLoads + u) * 1024), 16, off, at, 0, 0);
            }
        }
    };

    // ---- weights: a lane's 16 k of a column (l % 16) and sub-step, k = 16 (l / 16) .. + 15, are two operands
    const uint32_t left = p.n - n0 < BN ? p.n - n0 : BN;
    const uint64_t wbase = kInt4 ? static_cast<uint64_t>(n0 / 16u) * (p.k * 8u) : static_cast<uint64_t>(n0) * p.k;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.w) + wbase, 0, static_cast<int>(kInt4 ? (left + 15u) / 16u * (p.k * 8u) : left * p.k), 0x00020000);
    const uint32_t boff = kInt4 ? (lq >> 1) * 256u + lc * 16u + (lq & 1u) * 8u : lc * p.k + lq * 16u;
    const uint32_t bslab = kInt4 ? p.k * 8u : p.k * 16u;
    __amdgpu_buffer_rsrc_t rs = rw, ro = rw;                  // int4: parameters of a group of k and a column
    uint32_t poff = 0;
    if constexpr (kInt4) {
        const int bytes = static_cast<int>((p.k >> (5u + p.gs_shift)) * p.n * 2u);
        rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.scale), 0, bytes, 0x00020000);
        ro = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kOff ? p.offset : p.scale), 0, bytes, 0x00020000);
        poff = (n0 + lc) * 2u + (p.gs_shift == 0 ? (lq >> 1) * p.n * 2u : 0u);
    }
    struct Raw {
        u32x4 w[SUB][NJ];                                     // int4: the first two
        uint32_t sc[kParams], of[kParams];
    };
    auto fetch_one = [&](Raw& raw, uint32_t stage, int s, int j, auto parity) __attribute__((always_inline)) {
        constexpr int kPar = decltype(parity)::value;
        const uint32_t sub = sub0 + stage * SUB + s;
        if constexpr (kInt4) {
            const uint32_t pat = ((2u * sub) >> p.gs_shift) * p.n * 2u;
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rw, boff, sub * 512u + j * bslab, 0);
            raw.w[s][j][0] = v[0];
            raw.w[s][j][1] = v[1];
            if (Loads::params(kPar, s)) {
                raw.sc[s * NJ + j] = __builtin_amdgcn_raw_buffer_load_b16(rs, poff + j * 32u, pat, 0);
                if constexpr (kOff) raw.of[s * NJ + j] = __builtin_amdgcn_raw_buffer_load_b16(ro, poff + j * 32u, pat, 0);
            }
        } else {
            raw.w[s][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, boff, sub * 64u + j * bslab, 0));
        }
    };
    auto fetch = [&](Raw& raw, uint32_t stage, auto parity) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SUB; ++s)
#pragma unroll
            for (int j = 0; j < NJ; ++j) fetch_one(raw, stage, s, j, parity);
    };
    f16x2 csc[NJ], cof[NJ];                                   // int8: scale and offset belong to the column
    if constexpr (!kInt4) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t c = j * 16u + lc, gcol = n0 + (c < left ? c : left - 1u);
            csc[j] = as_h2((p.scale ? p.scale[gcol] : p.scale_bits) * 0x10001u);
            cof[j] = as_h2((kOff ? (p.scale ? p.offset[gcol] : p.offset_bits) : 0u) * 0x10001u);
        }
    }
    WqMasks mk = p.mk;
    asm volatile("" : "+v"(mk.exp_even), "+v"(mk.exp_odd));   // (an instruction takes one scalar operand)
    auto operand = [&](const Raw& raw, int s, int d, int j) __attribute__((always_inline)) {
        u32x4 h;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (kSum) {
                const uint32_t q = raw.w[s][j][d], src = c & 2 ? q >> 8 : q;
                h[c] = as_u32(c & 1 ? as_h2((src & mk.odd) | mk.exp_odd) - both(72.0f) : as_h2((src & mk.even) | mk.exp_even) - both(1032.0f));
            } else if constexpr (kInt4) {
                h[c] = pair_of_i4<kOff>(raw.w[s][j][d], c, as_h2(raw.sc[s * NJ + j] * 0x10001u), as_h2((kOff ? raw.of[s * NJ + j] : 0u) * 0x10001u), mk);
            } else {
                h[c] = pair_of_i8<kOff>(raw.w[s][j][2 * d + (c >> 1)], c & 1, csc[j], cof[j]);
            }
        }
        return __builtin_bit_cast(f16x8, h);
    };

    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[NI][NJ], part[kSum ? NI : 1][kSum ? NJ : 1], xs[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = zero;
    }
    f16x8 ones = {};
    if constexpr (kSum && kOff) {
        const u32x4 o = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
        ones = __builtin_bit_cast(f16x8, o);
        asm volatile("" : "+v"(ones));
    }
    uint32_t foff[2];                                         // the lane's places in a line block of 16 rows
#pragma unroll
    for (int d = 0; d < 2; ++d) foff[d] = wave * kStageBytes + lc * 128u + (((2u * lq + d) ^ wq_swizzle(lc)) << 4);

    // Stage `stage` lies in S and raw.
    auto step = [&](char* S, Raw& raw, uint32_t stage, auto parity) __attribute__((always_inline)) {
        // everything but the next stage's loads has arrived (the build looks the loads and counts over: check_matrix_asm.py)
        constexpr int kLeft = Loads::count(1 - decltype(parity)::value);
        __builtin_amdgcn_s_waitcnt(0x0F70 | (kLeft & 15) | ((kLeft >> 4) << 14));
        asm volatile("" ::: "memory");
        f16x8 af[SUB][2][NI];
#pragma unroll
        for (int s = 0; s < SUB; ++s)
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int i = 0; i < NI; ++i) af[s][d][i] = *reinterpret_cast<const f16x8*>(S + foff[d] + (s * NI + i) * 2048);
        __builtin_amdgcn_s_waitcnt(0xC07F);                   // the stage is read: its place takes the loads of the stage after next
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load_x(S, stage + 2u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            if (sub0 + stage * SUB + s < sub_end) {           // (uniform)
                constexpr int kPar = decltype(parity)::value;
                const bool first = ((kPar * SUB + s) & 1) == 0, last = !first;
                if constexpr (kSum && kOff) {
#pragma unroll
                    for (int d = 0; d < 2; ++d)
#pragma unroll
                        for (int i = 0; i < NI; ++i)
                            xs[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[s][d][i], ones, first && d == 0 ? zero : xs[i], 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        const f16x8 b = operand(raw, s, d, j);
#pragma unroll
                        for (int i = 0; i < NI; ++i) {
                            if constexpr (kSum) {
                                part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[s][d][i], b, first && d == 0 ? zero : part[i][j], 0, 0, 0);
                            } else {
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[s][d][i], b, acc[i][j], 0, 0, 0);
                            }
                        }
                    }
                }
                if constexpr (kSum) {
                    if (last) {                               // 128 k are done: they lie in one group
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            const float sc = half_bits_to_f32(raw.sc[s * NJ + j]), of = kOff ? half_bits_to_f32(raw.of[s * NJ + j]) : 0.0f;
#pragma unroll
                            for (int i = 0; i < NI; ++i)
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    const float v = kOff ? __builtin_fmaf(of, xs[i][r], part[i][j][r]) : part[i][j][r];
                                    acc[i][j][r] = __builtin_fmaf(sc, v, acc[i][j][r]);
                                }
                        }
                    }
                }
            }
        }
        fetch(raw, stage + 2u, parity);
        __builtin_amdgcn_sched_barrier(0);
    };

    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    Raw r0, r1;
    __builtin_amdgcn_sched_barrier(0);                        // (the first waits count these loads in this order)
    load_x(A0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(r0, 0, even);
    __builtin_amdgcn_sched_barrier(0);
    load_x(A1, 1);
    __builtin_amdgcn_sched_barrier(0);
    fetch(r1, 1, odd);
    __builtin_amdgcn_sched_barrier(0);
    for (uint32_t i = 0; i < stages; i += 2u) {
        step(A0, r0, i, even);
        step(A1, r1, i + 1u, odd);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                       // the loads past the end
    asm volatile("" ::: "memory");

    __syncthreads();

    // ---- the eight partial tiles meet in LDS and are added in wavefront order
    {
        float* const R = reinterpret_cast<float*>(wave < 4u ? A0 : A1) + (wave & 3u) * (BM * BN);
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) R[sum_place<BN>(i * 16u + 4u * lq + r, j * 16u + lc)] = acc[i][j][r];
    }
    __syncthreads();
    for (uint32_t e = tid; e < BM * BN / 4u; e += kWaves * 64u) {
        const uint32_t r = e / (BN / 4u), c = e % (BN / 4u) * 4u;
        const uint32_t place = sum_place<BN>(r, c);
        f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(A0) + place);
#pragma unroll
        for (uint32_t w = 1; w < kWaves; ++w)
            v += *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(w < 4u ? A0 : A1) + (w & 3u) * (BM * BN) + place);
        const uint32_t row = row0 + r, col = n0 + c;
        if (row >= p.m || col >= p.n) {
            continue;
        }
        const size_t idx = static_cast<size_t>(row) * p.n + col;
        if (p.wide_store) {
            if (p.out_f32) {
                *reinterpret_cast<f32x4*>(static_cast<float*>(p.y) + idx) = v;
            } else {
                *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.y) + idx) =
                    u32x2{f32_to_half_bits(v[0]) | (f32_to_half_bits(v[1]) << 16), f32_to_half_bits(v[2]) | (f32_to_half_bits(v[3]) << 16)};
            }
            continue;
        }
#pragma unroll
        for (uint32_t q = 0; q < 4u; ++q) {
            if (col + q < p.n) {
                if (p.out_f32) {
                    static_cast<float*>(p.y)[idx + q] = v[q];
                } else {
                    static_cast<uint16_t*>(p.y)[idx + q] = static_cast<uint16_t>(f32_to_half_bits(v[q]));
                }
            }
        }
    }
}

template <int BM, int BN>
void rows_launch(WqParams p, int kind, bool off, hipStream_t st)
{
    p.tiles_m = (p.m + BM - 1u) / BM;
    p.tiles_n = (p.n + BN - 1u) / BN;
    const uint32_t grid = (p.tiles_m * p.tiles_n + 7u) / 8u * 8u;
    auto go = [&](auto k) {
        constexpr int kKind = decltype(k)::value;
        off ? wq_rows_kernel<BM, BN, kKind, true><<<grid, kWaves * 64, 0, st>>>(p)
            : wq_rows_kernel<BM, BN, kKind, false><<<grid, kWaves * 64, 0, st>>>(p);
    };
    switch (kind) {
        case kInt4Weight: go(std::integral_constant<int, kInt4Weight>{}); break;
        case kInt4Sum:
            go(std::integral_constant<int, kInt4Sum>{});
            break;
        default: go(std::integral_constant<int, kInt8Weight>{}); break;
    }
}

}  // namespace

namespace {

// What a workgroup of each shape takes at k = 1024 to 14336 on an otherwise busy chip (us; least squares over 360 random calls,
// 5 to 2000 rows, nine tenths within 12 %): once, and per stage of its wavefronts.  int8 takes longer: a lane's 16 bytes are a quarter
// of a 64-byte run of its column, where int4 comes packed.
struct RowsShape {
    uint32_t bm, bn;
    double round4, stage4, round8, stage8;
};
constexpr RowsShape kShapes[] = {{16, 16, 3.00, 0.880, 4.48, 1.34}, {32, 16, 2.20, 0.745, 2.86, 1.06}, {32, 32, 2.80, 0.990, 4.00, 1.53},
                                 {64, 16, 1.75, 0.620, 2.44, 0.82}, {64, 32, 2.30, 0.745, 3.31, 1.05}, {64, 64, 3.30, 1.100, 5.13, 1.51}};

// the shape that is expected to be fastest; its time
int best_shape(uint32_t m, uint32_t n, uint32_t k, bool int4, double& us)
{
    const uint32_t cus = device_compute_units(), unit = int4 ? 2u : 1u;
    auto up = [](uint64_t a, uint64_t b) { return (a + b - 1u) / b; };
    int at = 0;
    us = 1e30;
    for (int i = 0; i < static_cast<int>(sizeof(kShapes) / sizeof(kShapes[0])); ++i) {
        const RowsShape& s = kShapes[i];
        const uint64_t tiles = up(m, s.bm) * up(n, s.bn);
        const uint64_t stages = up(up(k / 64u / unit, kWaves) * unit, 64u / s.bm);
        const double t = up(tiles, cus) * (int4 ? s.round4 + s.stage4 * stages : s.round8 + s.stage8 * stages);
        if (tiles < (1ull << 31) - 8u && t < us) {
            us = t;
            at = i;
        }
    }
    us += int4 ? 1.35 : 1.0;
    return at;
}

}  // namespace

double wq_rows_estimate(uint32_t m, uint32_t n, uint32_t k, bool int4)
{
    double us;
    best_shape(m, n, k, int4, us);
    return us;
}

bool wq_rows_ahead(const WqParams& p, bool int4, bool sum, bool has_offset, double other_us, hipStream_t st)
{
    if (p.k > kWqMaxK) {
        return false;
    }
    double us;
    const int at = best_shape(p.m, p.n, p.k, int4, us);
    // 5 % ahead, or the two are as good as each other.  int8 with up to 10 rows: 13 %, since the estimate is up to as much below
    // what these tiles take there (11 of 170 random calls were slower than in passes: 5 x 4736 x 8064 12.5 us in passes, 14.8
    // here, estimates 13.6 and 12.7)
    // int4 above 120 us: 15 %.  Many rounds of a full chip take up to a fifth longer than estimated (570 random calls, 12 of them slower
    // than on the large tiles, one with this: 179 x 10880 x 29824 157 us there, 189 here, estimates 175 and 166; 427 x 11776 x 12624 166
    // and 198).
    const double ahead = !int4 && p.m <= 10u ? 0.87 : int4 && us > 120.0 ? 0.85 : 0.95;
    if (us > ahead * other_us) {
        return false;
    }
    WqParams q = p;
    q.mk = WqMasks{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    q.wide_store = p.n % 4u == 0 && (reinterpret_cast<uintptr_t>(p.y) & (p.out_f32 ? 15u : 7u)) == 0 ? 1u : 0u;
    const int kind = int4 ? (sum ? kInt4Sum : kInt4Weight) : kInt8Weight;
    switch (at) {
        case 0: rows_launch<16, 16>(q, kind, has_offset, st); break;
        case 1: rows_launch<32, 16>(q, kind, has_offset, st); break;
        case 2: rows_launch<32, 32>(q, kind, has_offset, st); break;
        case 3: rows_launch<64, 16>(q, kind, has_offset, st); break;
        case 4: rows_launch<64, 32>(q, kind, has_offset, st); break;
        default: rows_launch<64, 64>(q, kind, has_offset, st); break;
    }
    return true;
}

}  // namespace ascq
