"""The kernels that calls choose, without a GPU (tests/routes.py): the sizes at which a rule was measured keep the faster side."""
import pytest

import test_gpu_matmul as sizes
import test_gpu_mx as mx_sizes
from ascq import _abi as abi
from routes import route

DST, SRC, SCALE, OFFSET = 1 << 44, 1 << 20, 1 << 42, 1 << 43      # apart, aligned, never read


def quant(rows, n, src=abi.BF16, par=abi.BF16, fmt=abi.QDST_I8, mode=abi.CAST_RINT, policy=abi.PER_CHANNEL, compute=abi.COMPUTE_F32, src_at=SRC):
    d = dict(policy=policy, src_dtype=src, scale_dtype=par, compute=compute, round_mode=mode, offset_kind=abi.OFFSET_NONE, k_dim=1, m=rows, n=n,
             cal_count=rows * n, group_size=32, dst_format=fmt)
    launch, = route("ascq_quant", ("QuantDesc", d), DST, src_at, None if policy == abi.PER_TENSOR else SCALE, None, None)
    return launch


@pytest.mark.parametrize("rows,n", [(4000, 4096), (100000, 32), (40000, 128), (4000, 1024)])
@pytest.mark.parametrize("fmt,mode", [(abi.QDST_I8, abi.CAST_FLOOR), (abi.QDST_HIF8, abi.CAST_ROUND)])
def test_formats_without_a_kernel_of_their_own_hold_two_rows_per_lane(rows, n, fmt, mode):
    """quant_vec_kernel<source, parameters, arithmetic, kind, rows per lane, any address>: four rows cost two of seven wavefronts."""
    assert quant(rows, n, fmt=fmt, mode=mode).args[3:] == ("4", "2", "false")
    assert quant(100, n, fmt=fmt, mode=mode).args[3:] == ("4", "1", "false")
    assert quant(rows, n).args[3:] == ("0", "4", "false")


@pytest.mark.parametrize("rows,n,per_lane", [(8192, 32, "1"), (8193, 32, "4"), (30000, 32, "4"), (4000, 32, "1"), (16000, 64, "4"), (2047, 512, "1"), (2049, 512, "4"),
                                             (1024, 1024, "1"), (1025, 1024, "4"), (1, 2 ** 20, "1")])
def test_narrow_rows_come_one_to_a_lane_up_to_8192_wavefronts(rows, n, per_lane):
    """Up to 2^20 elements a lane holds one row, unless the rows are that many wavefronts: quantisers and dequantisation policies."""
    assert quant(rows, n).args[4] == per_lane
    d = dict(policy=abi.PER_TOKEN, src_format=abi.QDST_FP8_E4M3FN, scale_dtype=abi.BF16, dst_dtype=abi.BF16, compute=abi.COMPUTE_SCALE_T,
             k_dim=1, m=rows, n=n, cal_count=rows * n, group_size=32)
    launch, = route("ascq_antiquant_policy", ("AntiQuantPolicyDesc", d), DST, SRC, SCALE, None, None)
    assert launch.name == "antiquant_policy_vec_kernel" and launch.args[4] == per_lane


@pytest.mark.parametrize("cols", [193, 16])
def test_rows_whose_walk_passes_32_bits_run_one_element_per_lane(cols):
    last = 2 ** 32 - 1 - 65535 * 8                # (a width off 16 is as wide as the vectors take it)
    for rows, kernel in ((last, "antiquant_vec_kernel"), (last + 1, "antiquant_scalar_kernel"), (2 ** 32 - 1, "antiquant_scalar_kernel")):
        d = dict(src_dtype=abi.I8, dst_dtype=abi.F16, has_offset=0, per_tensor=1, k=rows, n=cols)
        launch, = route("ascq_antiquant", ("AntiQuantDesc", d), 1 << 52, SRC, None, None, None)
        assert launch.name == kernel and launch.grid_y >= 1


# widths and numbers of elements from which rows off the vectors' width or alignment are vectors all the same
@pytest.mark.parametrize("src,par,compute,fmt,width,elements,scalar_name", [
    (abi.F16, abi.F16, abi.COMPUTE_F16, abi.QDST_I8, 96, 1 << 17, "quant_f16_fast_kernel"),
    (abi.BF16, abi.BF16, abi.COMPUTE_F16, abi.QDST_I8, 192, 1 << 20, "quant_vec_kernel"),
    (abi.F32, abi.F32, abi.COMPUTE_F32, abi.QDST_I8, 192, 1 << 20, "quant_vec_kernel"),
    (abi.BF16, abi.BF16, abi.COMPUTE_F32, abi.QDST_FP8_E4M3FN, 384, 3 << 20, "quant_vec_kernel"),
    (abi.F32, abi.F32, abi.COMPUTE_F32, abi.QDST_HIF8, 384, 3 << 20, "quant_vec_kernel")])
def test_quantisers_of_odd_widths_are_vectors_where_wide_and_many(src, par, compute, fmt, width, elements, scalar_name):
    mode = abi.CAST_ROUND if fmt == abi.QDST_HIF8 else abi.CAST_RINT
    for n in (9, width - 1, width + 1, 2051):
        for rows in (13, -(-elements // n) - 1, -(-elements // n)):
            for policy in (abi.PER_CHANNEL, abi.PER_TENSOR):
                if rows < 1:
                    continue
                cols = rows * n if policy == abi.PER_TENSOR else n        # one row, or rows of 2048
                if cols % 8 == 0:
                    continue
                launch = quant(rows, n, src, par, fmt, mode, policy, compute)
                assert launch.name == (scalar_name if cols >= width and rows * n >= elements else "quant_scalar_kernel"), (rows, n, policy)
    # a width of whole vectors off their alignment
    for rows in (7, 2048):
        assert quant(rows, 2048, src, par, fmt, mode, compute=compute, src_at=SRC + 4).name == (scalar_name if rows == 2048 else "quant_scalar_kernel")


@pytest.mark.parametrize("int4", [False, True])
@pytest.mark.parametrize("dst,per_tensor,elements", [(abi.F16, 0, 1 << 20), (abi.F16, 1, 3 << 19), (abi.BF16, 0, 2 << 20), (abi.BF16, 1, 3 << 20)])
def test_antiquant_of_odd_widths_is_vectors_where_wide_and_many(dst, per_tensor, elements, int4):
    for n in (10, 190, 194, 2050):
        for rows in (13, -(-elements // n) - 1, -(-elements // n)):
            d = dict(src_dtype=abi.I4 if int4 else abi.I8, dst_dtype=dst, has_offset=1, per_tensor=per_tensor, k=rows, n=n)
            launch, = route("ascq_antiquant", ("AntiQuantDesc", d), DST, SRC, OFFSET, SCALE, None)
            assert launch.name == ("antiquant_vec_kernel" if n >= 192 and rows * n >= elements else "antiquant_scalar_kernel"), (rows, n)


@pytest.mark.parametrize("rows,n,kernel", [(378, 35, "dynq_generic_kernel"), (63, 191, "dynq_generic_kernel"), (1023, 191, "dynq_generic_kernel"),
                                           (1, 193, "dynq_row_kernel"), (1024, 65, "dynq_row_kernel"), (1024, 63, "dynq_generic_kernel"),
                                           (4095, 9, "dynq_generic_kernel"), (4096, 9, "dynq_row_kernel"), (5, 7, "dynq_generic_kernel"),
                                           (5000, 7, "dynq_generic_kernel"), (3, 16383, "dynq_row_kernel"), (5000, 16385, "dynq_generic_kernel")])
def test_dynamic_quantiser_of_odd_widths_is_vectors_where_wide_or_many(rows, n, kernel):
    launch, = route("ascq_dynamic_quant_per_token", abi.BF16, rows, n, DST, SCALE, SRC, None)
    assert launch.name == kernel


def test_dynamic_quantiser_of_whole_vectors_off_their_alignment_is_as_odd_widths():
    for n, at, kernel in ((40, DST, "dynq_row_kernel"), (40, DST + 1, "dynq_generic_kernel"), (192, DST + 1, "dynq_row_kernel")):
        launch, = route("ascq_dynamic_quant_per_token", abi.F16, 67, n, at, SCALE, SRC, None)
        assert launch.name == kernel


def half_matmul(entry, m, k, n, room=1 << 35, **kw):
    x, w, scale, offset, ws = 1 << 30, 1 << 36, 1 << 38, 1 << 39, 1 << 40
    if entry == "ascq_matmul_w8a16":
        d = ("W8A16Desc", dict(m=m, n=n, k=k, has_offset=1, out_dtype=abi.F16, **kw))
        return route(entry, d, 1 << 42, x, w, offset, scale, ws, room, None)
    d = ("W4A16Desc", dict(m=m, n=n, k=k, has_offset=1, **kw))
    if entry == "ascq_matmul_w4a16":
        return route(entry, d, 1 << 42, x, w, scale, offset, ws, room, None)
    return route(entry, d, 1 << 42, x, w, scale, offset, None)


@pytest.mark.parametrize("m,k,n,whole_k", [(5, 4736, 8064, False), (6, 5376, 14336, False), (8, 4736, 7488, False), (10, 5376, 3424, False),
                                           (9, 3072, 1280, False), (9, 7808, 3312, True), (14, 8448, 1376, True), (16, 8448, 1920, True), (30, 1920, 5312, True)])
def test_int8_passes_of_few_rows_stay_where_they_are_ahead(m, k, n, whole_k):
    first, *_ = half_matmul("ascq_matmul_w8a16", m, k, n, trans_b=1)
    assert first.name == ("wq_rows_kernel" if whole_k else "w8a16_nk_kernel")


@pytest.mark.parametrize("m,k,n,packed", [(8, 3072, 13920, False), (9, 3456, 9728, False), (5, 2944, 15104, False), (12, 6272, 6272, False),
                                          (17, 9600, 7744, False), (12, 8448, 13088, False), (16, 8448, 1920, True), (33, 2304, 1152, True),
                                          (64, 1792, 22496, True), (97, 4096, 27392, True)])
def test_int4_passes_of_few_rows_stay_where_they_are_ahead(m, k, n, packed):
    first, *_ = half_matmul("ascq_matmul_w4a16", m, k, n, group_size=128)
    assert first.name == ("pack_w4_tiles_kernel" if packed else "w4a16_tile_kernel")


@pytest.mark.parametrize("m,k,n,group,passes", [(5, 13568, 8544, 64, True), (5, 6784, 5680, 32, True), (8, 13440, 8800, 64, True), (8, 6784, 5680, 32, False),
                                                (16, 13440, 4000, 64, False), (5, 6784, 5680, 128, False)])
def test_packed_int4_in_many_groups_stays_in_passes_with_the_fewest_rows(m, k, n, group, passes):
    first, *_ = half_matmul("ascq_matmul_w4a16_packed", m, k, n, group_size=group)
    assert first.name == ("w4a16_packed_kernel" if passes else "wq_rows_kernel")


@pytest.mark.parametrize("m,k,n,group,whole_k", [(179, 10880, 29824, 128, False), (427, 11776, 12624, 64, False), (316, 7040, 25960, 128, False),
                                                 (513, 9088, 13920, 128, False), (216, 14080, 8960, 128, True), (141, 8064, 19472, 128, True)])
def test_long_int4_calls_stay_on_the_large_tiles_where_those_are_ahead(m, k, n, group, whole_k):
    launch, = half_matmul("ascq_matmul_w4a16_packed", m, k, n, group_size=group)
    assert launch.name == ("wq_rows_kernel" if whole_k else "wq_gemm_kernel")


# ---- the sizes of the GPU tests run the kernels that those tests name
def each(groups):
    return [(kernel, size) for kernel, members in groups.items() for size in members]


@pytest.mark.parametrize("kernel,size", each(sizes.W4_MANY_ROWS))
def test_packed_int4_tests_of_many_rows_run_the_tiles_they_name(kernel, size):
    launch, = half_matmul("ascq_matmul_w4a16_packed", *size[:3], group_size=size[3])
    assert launch.kernel.startswith(kernel)


@pytest.mark.parametrize("kernel,size", each(sizes.W4_PACKED_FIRST))
def test_int4_tests_of_many_rows_pack_and_run_the_tiles_they_name(kernel, size):
    first, then = half_matmul("ascq_matmul_w4a16", *size[:3], group_size=size[3])
    assert first.name == "pack_w4_tiles_kernel" and then.kernel.startswith(kernel)


@pytest.mark.parametrize("kernel,size", each(sizes.W8_MANY_ROWS))
def test_int8_tests_of_many_rows_run_the_tiles_they_name(kernel, size):
    launch, = half_matmul("ascq_matmul_w8a16", *size, trans_b=1)
    assert launch.kernel.startswith(kernel)


@pytest.mark.parametrize("tile,size", each(sizes.W4_WHOLE_K))
def test_int4_tests_of_whole_k_tiles_run_the_tiles_they_name(tile, size):
    """wq_rows_kernel<rows, columns, kind, offset>: kind 0 int4 per weight, 1 group sums (groups of whole 128 k), 2 int8"""
    for mode in (abi.W4A16_PER_WEIGHT, abi.W4A16_GROUP_SUM):
        launch, = half_matmul("ascq_matmul_w4a16_packed", *size[:3], group_size=size[3], mode=mode)
        kind = 1 if mode == abi.W4A16_GROUP_SUM and size[3] % 128 == 0 else 0
        if not tile and kind == 0:
            assert launch.kernel.startswith("wq_gemm_kernel<128, 128, ")
        else:
            assert launch.kernel.startswith("wq_rows_kernel<%d, %d, %d, " % ((tile or (64, 64)) + (kind,)))


def test_int4_tests_of_whole_k_tiles_cover_every_tile_in_both_forms():
    for per_weight in (True, False):
        reached = {tile for tile, size in each(sizes.W4_WHOLE_K) if per_weight or size[3] % 128 == 0}
        assert {(16, 16), (32, 16), (32, 32), (64, 16), (64, 32), (64, 64)} <= reached


@pytest.mark.parametrize("tile,size", each(sizes.W8_WHOLE_K))
def test_int8_tests_of_whole_k_tiles_run_the_tiles_they_name(tile, size):
    first, *_ = half_matmul("ascq_matmul_w8a16", *size, trans_b=1)
    assert first.kernel.startswith("wq_rows_kernel<%d, %d, 2, " % tile if tile else "w8a16_nk_kernel")


@pytest.mark.parametrize("at_once,size", each(sizes.LOAD_RULE))
def test_load_rule_tests_run_the_form_they_name(at_once, size):
    m, n, kind, k = size
    if kind == "int4":
        last, = half_matmul("ascq_matmul_w4a16_packed", m, k, n, group_size=128)
    else:
        *_, last = half_matmul("ascq_matmul_w8a16", m, k, n, trans_b=int(k % 128 == 0))
    if at_once is None:
        assert last.kernel.startswith("wq_rows_kernel<64, 64, ")
    else:
        assert last.kernel.startswith("wq_gemm_kernel<128, 128, ") and last.args[4] == str(at_once).lower()


@pytest.mark.parametrize("kind,m,k,n", sizes.SMALL_WORKSPACE)
def test_workspaces_too_small_for_the_weights_run_passes(kind, m, k, n):
    small, whole = sizes.passes_workspace(kind, m, k, n)
    entry, kw = "ascq_matmul_" + kind, {"group_size": 128} if kind == "w4a16" else {}
    for room, kernels in ((whole, {"pack_w4_tiles_kernel", "transpose_i8_kernel"}), (small, {"w4a16_tile_kernel", "w8a16_tile_kernel"})):
        first, *_ = half_matmul(entry, m, k, n, room=room, **kw)
        assert first.name in kernels


def group_matmul(counts, k, n, nz=False, spare=0, out=abi.F16, act=abi.MM_ACT_NONE):
    mm = dict(m=sum(counts) + spare, n=n, k=k, out_dtype=out, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32, has_tok_scale=1,
              activation=act, act_beta=1.0, b_format=abi.MM_B_NZ if nz else abi.MM_B_ND)
    d = ("GroupMatmulDesc", dict(mm=("MatmulDesc", mm), groups=len(counts), group_list_kind=abi.GROUP_LIST_COUNTS))
    launch, = route("ascq_group_matmul_w8a8", d, 1 << 42, 1 << 30, 1 << 36, None, 1 << 38, 1 << 39, 1 << 40, None)
    return launch


@pytest.mark.parametrize("counts,long_k", sizes.GROUP_REMAINDERS)
@pytest.mark.parametrize("nz", [False, True])
def test_group_remainder_tests_cross_the_rule_that_names_the_instruction(counts, long_k, nz):
    forms = {above: {group_matmul(counts, k, sizes.GROUP_WIDE, nz).kernel for k in (256, 384, 1280, 1408, 2432, 2560, 3072, 3200) if (k >= long_k) == above}
             for above in (False, True)}
    assert len(forms[False]) == len(forms[True]) == 1 and forms[False] != forms[True]
    assert all(kernel.startswith("gemm_dma_group_kernel<") for kernel, in forms.values())
    assert group_matmul(counts, 1408, 544, nz).name == "gemm_group_ring_kernel"


@pytest.mark.parametrize("counts", sizes.GROUP_EDGES)
def test_group_edge_tests_run_both_kernels(counts):
    for n, kernel in ((520, "gemm_group_ring_kernel"), (sizes.GROUP_EDGES_WIDE, "gemm_dma_group_kernel")):
        assert group_matmul(counts, 256, n, spare=8, out=abi.BF16).name == kernel


def mx_matmul(m, n, k, fa, fb, scale_k, out=abi.F32):
    d = ("MxDesc", dict(m=m, n=n, k=k, scale_k=scale_k, a_format=fa, b_format=fb, out_dtype=out, has_bias=0))
    return route("ascq_matmul_mx", d, 1 << 42, 1 << 30, 1 << 33, 1 << 36, 1 << 37, None, 1 << 44, 1 << 40, None)[-1]


@pytest.mark.parametrize("fa,fb", [(mx_sizes.E4, mx_sizes.E4), (mx_sizes.E5, mx_sizes.E4), (mx_sizes.E5, mx_sizes.E5), (mx_sizes.F2, mx_sizes.F2)])
@pytest.mark.parametrize("steps", [1, 2, 5, 8])
def test_mx_comparisons_of_ring_and_large_tiles_run_both(fa, fb, steps):
    k = steps * (256 if fa == mx_sizes.F2 else 128)
    scale_k = max(16, (k // 32 + 7) // 8 * 8)
    assert mx_matmul(4100, 2344, k, fa, fb, scale_k).name == "mx_tile_kernel"
    for tile, m in mx_sizes.RING_AND_TILES.items():
        assert mx_matmul(m, 2344, k, fa, fb, scale_k).kernel.startswith("mx_ring_kernel<%d, %d, " % tile)


# rows, columns: the tile of test_mx_ring_tiles (k is 128 or 256 times 1 to 17)
@pytest.mark.parametrize("m,n,tile", [(131, 2801, (64, 64)), (449, 2530, (128, 64)), (700, 2999, (128, 128))])
def test_mx_ring_tests_run_the_tiles_they_name(m, n, tile):
    for fa, fb in ((mx_sizes.E4, mx_sizes.E5), (mx_sizes.F2, mx_sizes.F2)):
        for steps in (1, 2, 3, 6, 9, 17):
            k = steps * (256 if fa == mx_sizes.F2 else 128)
            assert mx_matmul(m, n, k, fa, fb, max(16, (k // 32 + 7) // 8 * 8)).kernel.startswith("mx_ring_kernel<%d, %d, " % tile)


E4, F2, F1 = mx_sizes.E4, mx_sizes.F2, mx_sizes.F1


# measured ahead by 8 % to six times
@pytest.mark.parametrize("m,n,k,fa,fb,kernel", [(2005, 9032, 256, F1, F2, "mx_tile_kernel"), (3682, 2820, 256, F2, F1, "mx_tile_kernel"),
                                                (971, 6737, 256, F1, F2, "mx_tile_kernel"), (66, 8240, 12032, F2, F1, "mx_decode_kernel"),
                                                (511, 1228, 8960, F1, F2, "mx_decode_kernel"), (230, 14080, 6912, F2, F1, "mx_ring_kernel"),
                                                (952, 558, 3328, F2, E4, "mx_decode_kernel"), (1411, 400, 3584, F2, E4, "mx_decode_kernel"),
                                                (326, 7783, 2560, E4, F1, "mx_ring_kernel")])
def test_mx_pairs_with_a_widened_operand_run_the_kernel_that_is_ahead(m, n, k, fa, fb, kernel):
    assert mx_matmul(m, n, k, fa, fb, max(16, (k // 32 + 7) // 8 * 8), abi.BF16).name == kernel


@pytest.mark.parametrize("counts,k,n,act,ring", [([1, 1], 128, 8736, abi.MM_ACT_SWIGLU, False), ([9, 2], 768, 11520, abi.MM_ACT_SWIGLU, False),
                                                 ([3, 1, 2, 1], 640, 4512, abi.MM_ACT_SWIGLU, False), ([18, 2], 384, 10912, abi.MM_ACT_NONE, False),
                                                 ([35, 26], 1024, 13536, abi.MM_ACT_SWIGLU, True), ([20, 10, 6, 4], 512, 4384, abi.MM_ACT_FASTER_GELU, True),
                                                 ([10] * 8, 256, 2272, abi.MM_ACT_NONE, True), ([93, 80, 60, 49], 640, 2944, abi.MM_ACT_NONE, True)])
def test_few_rows_of_few_groups_with_a_short_k_stay_off_the_ring(counts, k, n, act, ring):
    launch = group_matmul(counts, k, n, out=abi.BF16, act=act)
    assert launch.kernel.startswith("gemm_group_ring_kernel<64, 128, " if ring else "gemm_dma_group_kernel<")


@pytest.mark.parametrize("fa,fb", [(E4, E4), (F2, F2), (E4, F2), (F2, F1)])
def test_mx_rows_whose_offsets_pass_32_bits_leave_the_tiles(fa, fb):
    """The tiles and the ring address scale bytes by 32 bits from a's or b's first row, operands from a tile's; the few-row kernel by 64."""
    for m, n in ((128, 3000), (3000, 128), (700, 2999), (4100, 2344)):
        rows = max(m, n)
        last = (2 ** 32 - 1) // rows // 8 * 8            # the longest scale rows (in eights) that 32 bits reach
        assert mx_matmul(m, n, 1024, fa, fb, 64).name != "mx_elementwise_kernel"
        assert mx_matmul(m, n, 1024, fa, fb, last).kernel == mx_matmul(m, n, 1024, fa, fb, 64).kernel
        launch = mx_matmul(m, n, 1024, fa, fb, last + 8)
        assert launch.name == "mx_decode_kernel"
        if fa == E4 == fb:
            assert launch.args[4] == "false"             # as for any shape that the tiles do not take
    row = 1 << (25 if fa == fb == F2 else 24)            # values of a row of 2^24 bytes, the longest that 256 rows of 32-bit offsets hold
    assert mx_matmul(64, 4000, row, fa, fb, row // 32).name == "mx_tile_kernel"
    assert mx_matmul(64, 4000, row + 256, fa, fb, row // 32 + 8).name == "mx_elementwise_kernel"
