// Grouped int8 matmul on the direct-to-LDS tiles of matmul_w8a8_tile.h.
#include "matmul_w8a8_tile.h"

namespace ascq {
namespace {

// Rows [off, end) of group g (clipped to m); false when the group owns none.  `off` is carried from group to group.
__device__ __forceinline__ bool group_rows(const GemmParams& p, uint32_t g, int64_t& off, uint32_t& first, uint32_t& end)
{
    const int64_t v = p.group_list[g];
    const int64_t cnt = p.group_list_kind == ASCQ_GROUP_LIST_PREFIX_SUM ? v - off : v;
    if (cnt <= 0) {
        return false;
    }
    const int64_t begin = off;
    off += cnt;
    const int64_t stop = off > static_cast<int64_t>(p.m) ? static_cast<int64_t>(p.m) : off;
    first = static_cast<uint32_t>(begin);
    end = static_cast<uint32_t>(stop);
    return stop > begin;
}

// Row tiles of a group: `big` tiles of 256 rows (a remainder of more than 128 rows is one of them) and at most one
// small tile of 128 rows for a shorter remainder.
__device__ __forceinline__ void group_row_tiles(uint32_t rows, uint32_t& big, uint32_t& small)
{
    const uint32_t rem = rows & 255u;
    big = (rows >> 8) + (rem > 128u ? 1u : 0u);
    small = (rem != 0u && rem <= 128u) ? 1u : 0u;
}

// One phase of the grouped kernel's plan (see gemm_dma_group_kernel): the workgroup's ids that fall into it.
template <uint32_t phase, int kForm>
__device__ __forceinline__ void gemm_dma_group_phase(const GemmParams& p, const uint32_t* PLAN, const Stage& S0, const Stage& S1,
                                                     float* TS)
{
    for (uint32_t id = blockIdx.x;; id += gridDim.x) {
        const uint32_t tiles_n = p.tiles_n;
        const uint32_t big_tiles = __builtin_amdgcn_readfirstlane(PLAN[0]);
        const uint32_t small_tiles = __builtin_amdgcn_readfirstlane(PLAN[1]);
        const uint32_t wide = __builtin_amdgcn_readfirstlane(PLAN[2]);
        const uint32_t col_narrow = wide * 256u;
        const uint32_t narrow = col_narrow < p.n ? (p.n - col_narrow + 127u) / 128u : 0u;
        const uint32_t count0 = big_tiles * wide, count1 = big_tiles * narrow, count2 = small_tiles * tiles_n;
        const uint32_t first1 = (count0 + 7u) & ~7u, first2 = first1 + ((count1 + 7u) & ~7u);
        const uint32_t first = phase == 0 ? 0u : phase == 1 ? first1 : first2;
        const uint32_t count = phase == 0 ? count0 : phase == 1 ? count1 : count2;
        const uint32_t cols = phase == 0 ? wide : phase == 1 ? narrow : tiles_n;
        if (id < first) {
            continue;  // an id of an earlier phase
        }
        if (id >= first + ((count + 7u) & ~7u)) {
            break;
        }
        const uint32_t t = xcd_remap(id - first, count);
        if (t >= count) {
            continue;  // padding of the phase
        }
        TilePlace at{0, 0, 0, nullptr, 0};
        {
            uint32_t base = 0;
            int64_t off = 0;
            for (uint32_t g = 0; g < p.groups; ++g) {
                uint32_t first, end, big, small;
                if (!group_rows(p, g, off, first, end)) {
                    continue;
                }
                group_row_tiles(end - first, big, small);
                const uint32_t mine = phase == 2 ? small : big;
                if (t >= base + mine * cols) {
                    base += mine * cols;
                    continue;
                }
                const uint32_t local = t - base;
                const uint32_t tn = local / mine, tr = local - tn * mine;
                at.row0 = first + (phase == 2 ? ((end - first) >> 8) * 256u : tr * 256u);
                at.row_end = end;
                at.n0 = phase == 1 ? col_narrow + tn * 128u : tn * 256u;
                at.b = p.b + static_cast<size_t>(g) * p.k * p.n;
                at.chan_off = static_cast<size_t>(g) * p.n;
                break;
            }
        }
        if (at.b == nullptr) {
            continue;
        }
        if constexpr (phase == 0) {
            gemm_dma_tile_at<256, 256, false, true, 0, kForm>(p, at, 0u, TS, S0, S1);
        } else if constexpr (phase == 1) {
            gemm_dma_tile_at<256, 128, false, true, 0, kForm>(p, at, 0u, TS, S0, S1);
        } else if (at.row_end - at.row0 <= 64u) {  // uniform: a remainder of at most 64 rows
            gemm_dma_tile_at<64, 256, false, true, 0, kForm>(p, at, 0u, TS, S0, S1);
        } else {
            gemm_dma_tile_at<128, 256, false, true, 0, kForm>(p, at, 0u, TS, S0, S1);
        }
        __syncthreads();  // the next tile's loads and token scales overwrite what slower wavefronts may still read
    }
}

// The grouped matmul in one launch of persistent workgroups, one per compute unit.  Every workgroup reads the group
// list and derives the same plan from it:
//   phase 0: the big row tiles x the first `wide` 256-wide tile columns, as many as fill whole rounds of the chip;
//   phase 1: the big row tiles x the remaining columns as 256 x 128 tiles (the last, partial round in half-size pieces);
//   phase 2: the groups' short remainders (at most 128 rows) as 128 x 256 tiles (64 x 256 up to 64 rows), cheapest last.
// Tile ids run through the phases in this order (each phase padded to a multiple of 8 ids, so that id mod 8 stays the
// XCD of the workgroup that takes it); workgroup w takes ids w, w + gridDim.x, ...  Inside a phase the tiles are
// ordered group by group, column by column, the row tiles of a column adjacent, and an XCD takes a contiguous share:
// about one group per XCD, whose rows of A stay in that L2 while each B tile is fetched once for the row tiles that
// run side by side.  The group sizes are known only on the device, so a launch sized by the host for the worst case
// would consist mostly of workgroups with nothing to do; the loop has none.  gridDim.x must be a multiple of 8;
// p.tiles_n = 256-wide tile columns of the whole matrix.
template <int kForm>
__global__ __launch_bounds__(kThreads, 1) void gemm_dma_group_kernel(GemmParams p)
{
    ASCQ_DMA_STAGES(kForm, 256, 256);
    __shared__ __attribute__((aligned(16))) float TS[256];
    uint32_t n_big = 0, n_small = 0;
    {
        int64_t off = 0;
        for (uint32_t g = 0; g < p.groups; ++g) {
            uint32_t first, end, big, small;
            if (group_rows(p, g, off, first, end)) {
                group_row_tiles(end - first, big, small);
                n_big += big;
                n_small += small;
            }
        }
    }
    // The plan is parked in LDS and re-read per tile: held in scalar registers across the tile bodies it would push
    // the compiler into spilling them.
    __shared__ uint32_t PLAN[4];
    {
        const uint32_t units = n_big * p.tiles_n + (n_small * p.tiles_n + 1u) / 2u;  // work in 256 x 256 tiles
        uint32_t wide = n_big ? units / gridDim.x * gridDim.x / n_big : 0u;
        if (wide > p.tiles_n) {
            wide = p.tiles_n;
        }
        if (threadIdx.x == 0) {
            PLAN[0] = n_big;
            PLAN[1] = n_small;
            PLAN[2] = wide;
        }
        __syncthreads();
    }
    // One loop per phase (a workgroup's ids ascend, so it passes through the phases in order anyway): each loop holds
    // one tile shape's code and registers.
    gemm_dma_group_phase<0, kForm>(p, PLAN, S0, S1, TS);
    gemm_dma_group_phase<1, kForm>(p, PLAN, S0, S1, TS);
    gemm_dma_group_phase<2, kForm>(p, PLAN, S0, S1, TS);
}

}  // namespace

int launch_gemm_dma_group(GemmParams& p, hipStream_t st)
{
    const int ring = gemm_group_ring_shape(p);
    if (ring >= 0) {
        return launch_gemm_group_ring(p, ring, st);
    }
    const uint32_t tiles_n = (p.n + 255u) / 256u;
    // The group sizes are on the device; the kernel plans its tiles there.  One persistent workgroup per compute
    // unit (a multiple of 8, so that a workgroup's id mod 8 is its XCD), fewer when no group list over m rows
    // can need that many tiles: big row tiles hold more than 128 rows each, at most m / 256 + groups of them, and
    // every group adds at most one short remainder.
    const uint32_t big = p.m / 129u < p.m / 256u + p.groups ? p.m / 129u : p.m / 256u + p.groups;
    const uint32_t small = p.groups < p.m ? p.groups : p.m;
    const uint64_t most = static_cast<uint64_t>(big) * 2u * tiles_n + static_cast<uint64_t>(small) * tiles_n + 24u;
    uint32_t wgs = device_compute_units() / 8u * 8u;
    if (wgs == 0u) {
        wgs = 8u;
    }
    if (most < wgs) {
        wgs = static_cast<uint32_t>((most + 7u) / 8u * 8u);
    }
    p.tiles_m = big + small;
    p.tiles_n = tiles_n;
    if (plan_recording()) {
        plan_note(ASCQ_MM_KERNEL_DMA_256, 256, 256, BK, wgs, 1, 2u * (256u * BK + BK * 256u) + 256u * 4u, 0);
        return ASCQ_OK;
    }
    // The 16 x 16 x 64 form's loads have one and a half K steps to arrive, but a tile starts with two stages of them: it
    // takes long sums, shorter ones the more rows a group has.  Time of the 16 x 16 x 64 kernel over the 32 x 32 x 32 one's,
    // geometric means of random calls with up to 128 / 129 to 256 / more rows per group: k = 256 1.14 / 1.05 / 1.05, 1024 1.05 / 1.03 /
    // 0.99, 1280 1.02 / 1.02 / 0.98, 1408 1.02 / 0.98 / 0.99, 1536 1.03 / 0.98 / 0.96, 2048 0.99 / 0.97 / 0.95, 2560 0.94 / 0.95 / 0.94,
    // 3584 0.90 / 0.89 / 0.91.  (Big tiles in the one form and remainders in the other were ahead of both nowhere by more than 1 %.)
    const uint64_t rows = p.m, groups = p.groups;
    const uint32_t long_k = rows > 256u * groups ? 1280u : rows > 128u * groups ? 1408u : 2560u;
    if (p.k % BK != 0) {
        gemm_dma_group_kernel<k32Ragged><<<wgs, kThreads, 0, st>>>(p);
    } else if (gemm_half_output(p) && p.k >= long_k) {
        gemm_dma_group_kernel<k16><<<wgs, kThreads, 0, st>>>(p);
    } else {
        gemm_dma_group_kernel<k32><<<wgs, kThreads, 0, st>>>(p);
    }
    return launch_status("ascq_group_matmul_w8a8");
}

}  // namespace ascq
