// int8 matmul of medium size: small tiles with a ring of LDS stages.
//
// What bounds these calls is the way of the operands into the LDS, and its latency: 256 x 256 tiles leave most of the chip
// idle, and a loop that waits for all of its loads at every K step takes 0.8 to 1.3 us for one, whatever its size.  Here
// a workgroup (8 wavefronts, v_mfma_i32_16x16x64_i8) owns a tile small enough for most compute units to have one, and the 128 KiB
// or so of stages that its loads fill hold 4 to 8 K steps: a load has kStages - 1/2 steps to arrive, and a step waits only for
// the next one's.  A step's operands are read from the LDS behind the matrix instructions of the step before.  No K split, so no
// int32 partial tiles and no second launch.  A last, partial K step and the steps past
// the end are loads whose offset lies past the buffer: zeros arrive.
// In us with the quantiser, split or large tiles and this: 729 x 4304 x 1152 27.8 and 19.2, 600 x 4096 x 4096 47.4 and 27.8, 1024 x
// 11008 x 4096 103 and 64.  What is left: a step of 64 x 64 takes 0.19 us without the bytes of its loads (the barrier, ten LDS
// reads and two loads per wavefront), one of 128 x 128 0.46 with nothing but loads (what is in flight over the latency of an L2 miss).
#include "matmul_w8a8_tile.h"

namespace ascq {
namespace {

template <int BM, int BN, int kStages, int kB, int kForm>
__global__ __launch_bounds__(kThreads, 1) void gemm_ring_kernel(GemmParams p)
{
    constexpr int kBytes = (BM + BN) * BK, kOther = 16;
    // (an array per stage: the compiler tells at most eight targets of such loads apart; one that nothing reads takes no space)
    __shared__ __attribute__((aligned(1024))) char L0[kBytes], L1[kBytes], L2[kBytes], L3[kBytes],
        L4[kStages > 4 ? kBytes : kOther], L5[kStages > 5 ? kBytes : kOther], L6[kStages > 6 ? kBytes : kOther], L7[kStages > 7 ? kBytes : kOther];
    __shared__ __attribute__((aligned(16))) float TS[BM];
    const uint32_t t = xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n);
    if (t >= p.tiles_m * p.tiles_n) {
        return;
    }
    uint32_t ms, tn;
    band_order(t, p.tiles_m, p.tiles_n, ms, tn);
    const TilePlace at{ms * BM, p.m, tn * BN, p.b, 0};
    char* const all[8] = {L0, L1, L2, L3, L4, L5, L6, L7};
    char* ring[kStages];
    static_for<kStages>([&](auto i) { ring[decltype(i)::value] = all[decltype(i)::value]; });
    gemm_dma_tile_at<BM, BN, false, false, kB, kForm>(p, at, 0u, TS, ring);
}

template <int BM, int BN, int kStages, int kB>
void run_ring(const GemmParams& q, uint32_t grid, hipStream_t st)
{
    if (gemm_half_output(q) && q.epi.activation != ASCQ_MM_ACT_SWIGLU && q.epi.scale_format == ASCQ_MM_SCALE_F32) {
        gemm_ring_kernel<BM, BN, kStages, kB, kRingHalf><<<grid, kThreads, 0, st>>>(q);
    } else {
        gemm_ring_kernel<BM, BN, kStages, kB, kRing><<<grid, kThreads, 0, st>>>(q);
    }
}

template <int BM, int BN, int kStages>
void run_ring(const GemmParams& p, int b_layout, hipStream_t st)
{
    GemmParams q = p;
    q.tiles_m = (p.m + BM - 1u) / BM;
    q.tiles_n = (p.n + BN - 1u) / BN;
    const uint32_t grid = (q.tiles_m * q.tiles_n + 7u) / 8u * 8u;
    if (b_layout == 2) {
        run_ring<BM, BN, kStages, 2>(q, grid, st);
    } else if (b_layout == 1) {
        run_ring<BM, BN, kStages, 1>(q, grid, st);
    } else {
        run_ring<BM, BN, kStages, 0>(q, grid, st);
    }
}

// The same for a grouped matmul: persistent workgroups that share out the tiles of all groups, group by group, inside a group column by
// column with the row tiles of a column adjacent.  The group sizes are on the device: lane g holds what group g owns (at most 64 groups),
// scans over the lanes give its rows and tiles.
// (Where these are taken, and what they measured: gemm_group_ring_shape.)
constexpr uint32_t kGroupLanes = 64;

template <int BM, int BN, int kStages, int kForm>
__global__ __launch_bounds__(kThreads, 1) void gemm_group_ring_kernel(GemmParams p)
{
    constexpr int kBytes = (BM + BN) * BK, kOther = 16;
    __shared__ __attribute__((aligned(1024))) char L0[kBytes], L1[kBytes], L2[kBytes], L3[kBytes],
        L4[kStages > 4 ? kBytes : kOther], L5[kStages > 5 ? kBytes : kOther], L6[kStages > 6 ? kBytes : kOther], L7[kStages > 7 ? kBytes : kOther];
    __shared__ __attribute__((aligned(16))) float TS[BM];
    const uint32_t g = threadIdx.x & 63u;
    uint32_t rows_end, tiles_end, first;
    {
        int64_t v = g < p.groups ? p.group_list[g] : 0;
        v = v < 0 ? 0 : (v > static_cast<int64_t>(p.m) ? static_cast<int64_t>(p.m) : v);
        const bool prefix = p.group_list_kind == ASCQ_GROUP_LIST_PREFIX_SUM;
        rows_end = static_cast<uint32_t>(v);
#pragma unroll
        for (uint32_t d = 1; d < 64u; d *= 2u) {  // rows up to this group's end: the largest prefix or the sum of the counts, at most m
            const uint32_t below = __shfl_up(rows_end, d, 64);
            const uint64_t sum = static_cast<uint64_t>(rows_end) + below;
            const uint32_t with = prefix ? (below > rows_end ? below : rows_end) : (sum < p.m ? static_cast<uint32_t>(sum) : p.m);
            rows_end = g >= d ? with : rows_end;
        }
        const uint32_t before = __shfl_up(rows_end, 1, 64);
        first = g == 0u ? 0u : before;
        tiles_end = (rows_end - first + BM - 1u) / BM;
#pragma unroll
        for (uint32_t d = 1; d < 64u; d *= 2u) {
            const uint32_t below = __shfl_up(tiles_end, d, 64);
            tiles_end += g >= d ? below : 0u;
        }
    }
    const uint32_t row_tiles = __builtin_amdgcn_readlane(tiles_end, 63), total = row_tiles * p.tiles_n;
    char* const all[8] = {L0, L1, L2, L3, L4, L5, L6, L7};
    char* ring[kStages];
    static_for<kStages>([&](auto i) { ring[decltype(i)::value] = all[decltype(i)::value]; });
    for (uint32_t id = blockIdx.x; id < (total + 7u) / 8u * 8u; id += gridDim.x) {
        const uint32_t t = xcd_remap(id, total);
        if (t >= total) {
            continue;  // whole workgroup (ids are rounded up to a multiple of 8)
        }
        // the first group whose tiles end past this one
        const uint32_t at_g = __builtin_ctzll(__builtin_amdgcn_ballot_w64(tiles_end * p.tiles_n > t));
        const uint32_t row0 = __builtin_amdgcn_readlane(first, at_g), end = __builtin_amdgcn_readlane(rows_end, at_g);
        const uint32_t mine = (end - row0 + BM - 1u) / BM;
        const uint32_t local = t - (__builtin_amdgcn_readlane(tiles_end, at_g) - mine) * p.tiles_n, tn = local / mine, tr = local - tn * mine;
        const TilePlace at{row0 + tr * BM, end, tn * BN, p.b + static_cast<size_t>(at_g) * p.k * p.n, static_cast<size_t>(at_g) * p.n};
        gemm_dma_tile_at<BM, BN, false, true, 0, kForm>(p, at, 0u, TS, ring);
        __syncthreads();  // the next tile's loads and token scales overwrite what slower wavefronts may still read
    }
}

template <int BM, int BN, int kStages>
void run_group_ring(GemmParams p, uint32_t wgs, hipStream_t st)
{
    p.tiles_n = (p.n + BN - 1u) / BN;
    if (gemm_half_output(p) && p.epi.activation != ASCQ_MM_ACT_SWIGLU) {
        gemm_group_ring_kernel<BM, BN, kStages, kRingHalf><<<wgs, kThreads, 0, st>>>(p);
    } else {
        gemm_group_ring_kernel<BM, BN, kStages, kRing><<<wgs, kThreads, 0, st>>>(p);
    }
}

}  // namespace

// The tile of a call and its time with the quantiser in front, in us: 8.5, then rounds of the chip times K steps times a step's
// time, which grows with the part f of the compute units that have a tile (the way to memory is shared).  Measured on 64 to 256 tiles at
// k = 2048 to 11008, weights packed or as [n, k]: 64 x 64 0.225; 128 x 64 0.29 .. 0.415; 128 x 128 0.44 .. 0.62.  As
// [k, n], whose rows a tile of 64 columns reads as half lines: 0.30; 0.36 .. 0.48; 0.48 .. 0.66.  (64 x 128 and 256 x 128 were ahead of these nowhere by
// more than 8 %.)
RingPlan gemm_ring_plan(uint32_t m, uint32_t n, uint32_t k, int b_layout)
{
    struct Shape {
        uint32_t bm, bn;
        double start, step[2], fill[2];  // [b_layout == 0]
    };
    static constexpr Shape kShapes[] = {{64, 64, 8.5, {0.225, 0.30}, {0.0, 0.0}},
                                        {128, 64, 8.5, {0.26, 0.33}, {0.155, 0.15}},
                                        {128, 128, 8.5, {0.38, 0.44}, {0.24, 0.22}}};
    const uint32_t steps = (k + BK - 1u) / BK, cus = device_compute_units();
    RingPlan best{0, 64, 64, 1e30};
    for (int i = 0; i < 3; ++i) {
        const Shape& s = kShapes[i];
        const uint64_t tiles = static_cast<uint64_t>((m + s.bm - 1u) / s.bm) * ((n + s.bn - 1u) / s.bn);
        const double step = s.step[b_layout == 0], fill = s.fill[b_layout == 0], rest = static_cast<double>(tiles % cus) / cus;
        const double rounds = static_cast<double>(tiles / cus) * (step + fill) + (rest > 0.0 ? step + fill * rest : 0.0);
        const double us = s.start + steps * rounds * (tiles > cus ? 1.05 : 1.0);
        if (us < best.us) {
            best = RingPlan{i, s.bm, s.bn, us};
        }
    }
    return best;
}

int launch_gemm_ring(const GemmParams& p, int shape, int b_layout, hipStream_t st)
{
    if (plan_recording()) {
        static constexpr uint32_t kTile[3][3] = {{64, 64, 8}, {128, 64, 6}, {128, 128, 4}};
        const uint32_t bm = kTile[shape][0], bn = kTile[shape][1];
        plan_note(ASCQ_MM_KERNEL_DMA_128, bm, bn, BK, ((p.m + bm - 1u) / bm * ((p.n + bn - 1u) / bn) + 7u) / 8u * 8u, 1,
                  kTile[shape][2] * (bm + bn) * BK + bm * 4u, 0);
        return ASCQ_OK;
    }
    switch (shape) {
    case 0: run_ring<64, 64, 8>(p, b_layout, st); break;
    case 1: run_ring<128, 64, 6>(p, b_layout, st); break;
    default: run_ring<128, 128, 4>(p, b_layout, st); break;
    }
    return launch_status("ascq_matmul_w8a8 (ring)");
}

// the most tiles that a group list over m rows can need
static uint64_t group_ring_tiles(const GemmParams& p, uint32_t bm, uint32_t bn)
{
    const uint64_t rows = (p.m + static_cast<uint64_t>(p.groups) * (bm - 1u)) / bm;
    return (rows < p.m ? rows : p.m) * ((p.n + bn - 1u) / bn);
}

// Offsets inside a tile fit 31 bits (of a fractal matrix, from its first column).
static bool gemm_group_ring_supported(const GemmParams& p)
{
    constexpr uint32_t kMost = 1u << 23;
    return p.groups <= kGroupLanes && p.k <= kMost && p.n <= kMost && p.m < (1u << 31) && (p.n % 16u == 0 || p.n >= 256u) &&
           (!p.b_nz || static_cast<uint64_t>(p.n) * p.k < (1ull << 31) - 256u);
}

// The largest tiles that no group list over m rows can turn into more than one round of the chip, smallest first: with a second round
// the tiles of matmul_w8a8_group.hip are ahead, which start a tile with less to wait for.  In us there and with 64 x 64, 64 x 128 and
// 128 x 128 tiles: 8 groups, 195 rows, k = 2688, n = 1536 25.9 and 12.6, 16.1, 19.0; 16, 30, 3712, 1824 29.8 and 25.4, 21.0, 23.4;
// 4, 907, 1024, 2080 14.6 and 19.4, 18.1, 12.9; 8, 472, 2304, 6784 32.2 and 46.0, 43.9, 36.5; -1: none of them.
// Nor do few rows of few groups with a short k take the 64 x 128 tiles, whose ring costs more to fill than they have to do (us there and
// here, 560 random calls: 2 groups, 2 rows, k = 128, n = 8736 5.6 and 7.4; 2, 11, 768, 11520 7.6 and 9.0; 4, 7, 640, 4512 7.7 and 8.6;
// ahead again 2, 61, 1024, 13536 12.3 and 11.0, with FasterGelu 4, 40, 512, 4384 8.8 and 7.8, and from 5 groups on).
int gemm_group_ring_shape(const GemmParams& p)
{
    static constexpr uint32_t kTile[3][2] = {{64, 64}, {64, 128}, {128, 128}};
    for (int i = 0; i < 3; ++i) {
        if (group_ring_tiles(p, kTile[i][0], kTile[i][1]) <= device_compute_units()) {
            const bool few = i == 1 && p.groups <= 4u && p.m <= 64u && p.k < (p.groups <= 2u ? 1024u : 704u) &&
                             p.epi.activation != ASCQ_MM_ACT_FASTER_GELU;
            return gemm_group_ring_supported(p) && !few ? i : -1;
        }
    }
    return -1;
}

int launch_gemm_group_ring(const GemmParams& p, int shape, hipStream_t st)
{
    static constexpr uint32_t kTile[3][3] = {{64, 64, 8}, {64, 128, 6}, {128, 128, 4}};
    const uint32_t bm = kTile[shape][0], bn = kTile[shape][1];
    const uint32_t wgs = static_cast<uint32_t>((group_ring_tiles(p, bm, bn) + 7u) / 8u * 8u);
    if (plan_recording()) {
        plan_note(ASCQ_MM_KERNEL_DMA_128, bm, bn, BK, wgs, 1, kTile[shape][2] * (bm + bn) * BK + bm * 4u, 0);
        return ASCQ_OK;
    }
    switch (shape) {
    case 0: run_group_ring<64, 64, 8>(p, wgs, st); break;
    case 1: run_group_ring<64, 128, 6>(p, wgs, st); break;
    default: run_group_ring<128, 128, 4>(p, wgs, st); break;
    }
    return launch_status("ascq_group_matmul_w8a8 (ring)");
}

}  // namespace ascq
