// Large-M int8 matmul on the direct-to-LDS tiles of matmul_w8a8_tile.h.
#include "matmul_w8a8_tile.h"

namespace ascq {
namespace {

// Second pass of the split-K path: sums the int32 partial tiles [split][m][n] in split order (integer addition: exact in
// any order) and applies the epilogue.  One lane = four consecutive columns.
__global__ __launch_bounds__(256) void splitk_sum_epilogue_kernel(GemmParams p)
{
    const size_t quads = static_cast<size_t>(p.m) * p.n / 4u;
    const size_t plane = static_cast<size_t>(p.m) * p.n;
    for (size_t qd = static_cast<size_t>(blockIdx.x) * 256u + threadIdx.x; qd < quads;
         qd += static_cast<size_t>(gridDim.x) * 256u) {
        const size_t idx = qd * 4u;
        i32x4 acc = *reinterpret_cast<const i32x4*>(p.partial + idx);
        for (uint32_t sp = 1; sp < p.k_splits; ++sp) {
            const i32x4 v = *reinterpret_cast<const i32x4*>(p.partial + sp * plane + idx);
            acc += v;
        }
        const size_t row = idx / p.n, col = idx % p.n;
        const float tok = p.epi.has_tok ? p.epi.tok_scale[row] : 1.0f;
        dispatch_out(p.epi, [&](auto tag) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                int32_t a = acc[c];
                if (p.epi.bias_kind == ASCQ_MM_BIAS_I32_PRE) {
                    a += static_cast<const int32_t*>(p.epi.bias)[col + c];
                }
                epilogue_store<decltype(tag)::value>(p.epi, row, col + c, a, load_channel_q(p.epi, col + c), tok,
                                                     load_bias_post(p.epi, col + c));
            }
        });
    }
}

}  // namespace

// Whole 16-byte pieces along k of both operands ([n, k], packed: its tiles of 64 k) or along n ([k, n], where a last tile
// moved left to end at n also starts its pieces at 8 bytes; it needs a whole tile's columns then).  A last partial K step
// is masked where it is loaded.
bool gemm_dma_supported(const GemmParams& p, int b_layout)
{
    if (p.k % (b_layout == 2 ? 64u : 16u) != 0 || p.n < 16u || !aligned16(p.a) || !aligned16(p.b)) {
        return false;
    }
    if (p.b_nz) {
        return p.k % BK == 0 && p.n % 32u == 0;
    }
    return p.n % 16u == 0 || (p.n % 8u == 0 && (b_layout != 0 || p.n >= 256u));
}

namespace {

void run_dma(int form, const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st)
{
    if (form == k32Ragged) {
        run_dma_ragged(p, l, b_layout, st);
    } else if (form == k16) {
        run_dma_long(p, l, b_layout, st);
    } else {
        run_dma<k32>(p, l, b_layout, st);
    }
}

}  // namespace

int launch_gemm_dma(GemmParams& p, hipStream_t st, int b_layout)
{
    uint32_t tiles_n = (p.n + 255u) / 256u;
    p.tiles_m = (p.m + 255u) / 256u;
    // Tile quantisation: when the last round of 256-wide tiles would fill less than half of the 256 CUs, its
    // columns are computed with 128-wide tiles, which finish that round in about half the time.
    uint32_t narrow_cols = 0;  // number of 256-wide column tiles handed to the 128-wide kernel
    const uint32_t total = p.tiles_m * tiles_n;
    const uint32_t rem = total % 256u;
    if (total > 256u && rem != 0 && rem <= 128u) {
        narrow_cols = (rem + p.tiles_m - 1) / p.tiles_m;
        if (narrow_cols > tiles_n) {
            narrow_cols = tiles_n;
        }
    }
    const uint32_t wide_cols = tiles_n - narrow_cols;
    if (plan_recording()) {
        constexpr uint32_t kLdsWide = 2u * (256u * BK + BK * 256u) + 256u * 4u;
        constexpr uint32_t kLdsNarrow = 2u * (256u * BK + BK * 128u) + 256u * 4u;
        const uint32_t wide_wg = (p.tiles_m * wide_cols + 7u) / 8u * 8u;
        const uint32_t narrow_tiles = narrow_cols ? (p.n - wide_cols * 256u + 127u) / 128u : 0u;
        const uint32_t narrow_wg = (p.tiles_m * narrow_tiles + 7u) / 8u * 8u;
        if (wide_cols) {
            plan_note(ASCQ_MM_KERNEL_DMA_256, 256, 256, BK, wide_wg, 1, kLdsWide, 0);
            if (narrow_cols) {
                plan_note_extra(128, narrow_wg);  // workgroups of the same launch
            }
        } else {
            plan_note(ASCQ_MM_KERNEL_DMA_256, 256, 128, BK, narrow_wg, 1, kLdsNarrow, 0);
        }
        return ASCQ_OK;
    }
    const int form = gemm_dma_form(p);
    if (wide_cols && narrow_cols) {
        // both tile shapes in one launch (narrow_cols is only ever non-zero for the plain matmul)
        const uint32_t col_begin = wide_cols * 256u;
        const uint32_t narrow_tiles_n = (p.n - col_begin + 127u) / 128u;
        const uint32_t wide_wgs = (p.tiles_m * wide_cols + 7u) / 8u * 8u;
        const uint32_t narrow_wgs = (p.tiles_m * narrow_tiles_n + 7u) / 8u * 8u;
        p.tiles_n = wide_cols;
        run_dma(form, p, DmaLaunch{DmaLaunch::kBoth, dim3(wide_wgs + narrow_wgs), col_begin, wide_wgs, narrow_tiles_n}, b_layout, st);
        return launch_status("ascq_matmul_w8a8");
    }
    if (wide_cols) {
        p.tiles_n = wide_cols;
        const uint32_t t = p.tiles_m * p.tiles_n;
        run_dma(form, p, DmaLaunch{DmaLaunch::kWide, dim3((t + 7u) / 8u * 8u), 0u, 0u, 0u}, b_layout, st);
    } else {
        p.tiles_n = (p.n + 127u) / 128u;
        const uint32_t t = p.tiles_m * p.tiles_n;
        run_dma(p.k % BK != 0 ? k32Ragged : k32, p, DmaLaunch{DmaLaunch::kNarrow, dim3((t + 7u) / 8u * 8u), 0u, 0u, 0u}, b_layout, st);
    }
    return launch_status("ascq_matmul_w8a8");
}

// Split factor of the 128 x 128 kernel: two workgroups per CU when the partial tiles are small next to the weights,
// one per CU otherwise; never more splits than K steps.
uint32_t gemm_dma_skinny_splits(uint32_t m, uint32_t n, uint32_t k)
{
    // Measured at k = 4096, n = 11008 (86 column tiles) with the weights coming from HBM: one row tile (m <= 128) is
    // fastest with 4 splits (17-25 us; 2 splits 21-25, 6 splits 25-32, none 30), two or more row tiles are fastest
    // with none (30-32 us for m = 160 .. 384 against 32-55 with 2): once the tiles alone cover most of the compute
    // units the int32 partial tiles, written and read back, cost more than the idle units.  Hence: no split from 160
    // tiles on, otherwise about 1.35 workgroups per compute unit, all resident at once (two fit a unit).
    const uint32_t tiles = ((m + 127u) / 128u) * ((n + 127u) / 128u);
    if (tiles >= 160u) {
        return 1u;
    }
    uint32_t s = 344u / tiles;
    const uint32_t steps = (k + BK - 1u) / BK;
    if (s > steps) s = steps;
    if (s > 16u) s = 16u;
    return s ? s : 1u;
}

// More than 512 rows: whether the 128 x 128 tiles, K split, are expected ahead of the 256 x 256 ones, which leave most of
// the chip idle on a narrow matrix.  In us: a 256 x 256 tile takes 1.3 per K step when most units have none; a split
// of 128 x 128 tiles 0.8 per K step, a launch of 4 and its int32 partial tiles, written and read back at 5 TB/s
// (729 rows, k = 4352, n = 1152, quantiser included: 52 us on 15 wide tiles, 26 us on 54 split in six; 532 rows, k = 3072,
// n = 512: 38.5 and 24.4 us).
bool gemm_dma_small_tiles(uint32_t m, uint32_t n, uint32_t k)
{
    const uint32_t wide = ((m + 255u) / 256u) * ((n + 255u) / 256u);
    const uint32_t splits = gemm_dma_skinny_splits(m, n, k);
    if (wide > 64u || splits < 2u) {
        return false;
    }
    const uint32_t steps = (k + BK - 1u) / BK;
    const double split_us = 4.0 + 0.8 * ((steps + splits - 1u) / splits) + static_cast<double>(splits) * m * n * 8.0 / 5e6;
    return split_us < 1.3 * steps;
}

// M up to a few hundred rows, or few tiles: 128 x 128 tiles, K split over blockIdx.y when a workspace of
// splits * m * n * 4 bytes (16-byte aligned) is given.  b_layout: 0 [k, n], 1 [n, k], 2 packed.
int launch_gemm_dma_skinny(GemmParams& p, void* workspace, size_t workspace_bytes, hipStream_t st, int b_layout)
{
    p.tiles_m = (p.m + 127u) / 128u;
    p.tiles_n = (p.n + 127u) / 128u;
    const uint32_t t = (p.tiles_m * p.tiles_n + 7u) / 8u * 8u;
    uint32_t splits = gemm_dma_skinny_splits(p.m, p.n, p.k);
    const size_t need = static_cast<size_t>(splits) * p.m * p.n * sizeof(int32_t);
    if (splits > 1 && (workspace == nullptr || workspace_bytes < need || !aligned16(workspace))) {
        splits = 1;
    }
    if (plan_recording()) {
        constexpr uint32_t kLds = 2u * (128u * BK + BK * 128u) + 128u * 4u;
        plan_note(ASCQ_MM_KERNEL_DMA_128, 128, 128, BK, t * splits, splits, kLds, splits > 1 ? need : 0);
        if (splits > 1) {
            plan_note(0, 0, 0, 0, 0, 0, 0, 0);  // the kernel that adds the partial tiles and applies the epilogue
        }
        return ASCQ_OK;
    }
    const int form = p.k % BK != 0 ? k32Ragged : k32;
    if (splits == 1) {
        run_dma(form, p, DmaLaunch{DmaLaunch::kSmall, dim3(t), 0u, 0u, 0u}, b_layout, st);
        return launch_status("ascq_matmul_w8a8");
    }
    p.k_splits = splits;
    p.partial = static_cast<int32_t*>(workspace);
    run_dma(form, p, DmaLaunch{DmaLaunch::kSplit, dim3(t, splits), 0u, 0u, 0u}, b_layout, st);
    int rc = launch_status("ascq_matmul_w8a8 (split-K)");
    if (rc != ASCQ_OK) {
        return rc;
    }
    size_t blocks = (static_cast<size_t>(p.m) * p.n / 4u + 255u) / 256u;
    if (blocks > 8192u) blocks = 8192u;
    splitk_sum_epilogue_kernel<<<static_cast<uint32_t>(blocks), 256, 0, st>>>(p);
    return launch_status("ascq_matmul_w8a8 (split-K epilogue)");
}

}  // namespace ascq
