"""The kernels that calls choose, without a GPU (tests/routes.py): the sizes at which a rule was measured keep the faster side."""
import pytest

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


def half_matmul(entry, m, k, n, **kw):
    x, w, scale, offset, ws = 1 << 30, 1 << 36, 1 << 38, 1 << 39, 1 << 40
    if entry == "ascq_matmul_w8a16":
        d = ("W8A16Desc", dict(m=m, n=n, k=k, has_offset=1, out_dtype=abi.F16, **kw))
        return route(entry, d, 1 << 42, x, w, offset, scale, ws, 1 << 35, None)
    d = ("W4A16Desc", dict(m=m, n=n, k=k, has_offset=1, **kw))
    if entry == "ascq_matmul_w4a16":
        return route(entry, d, 1 << 42, x, w, scale, offset, ws, 1 << 35, None)
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
