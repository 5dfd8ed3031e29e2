"""How the element-wise kernels share out a matrix, at the last counts that 32 bits hold: no GPU."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from ascq import _abi as abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOP = 1 << 32


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    """row_walk.h behind C functions, built with the host compiler alone"""
    where = tmp_path_factory.mktemp("row_walk")
    src = where / "t.cpp"
    src.write_text('#include "row_walk.h"\n'
                   'extern "C" {\n'
                   'uint32_t lanes(uint32_t n) { return ascq::row_lanes(n); }\n'
                   'uint32_t fits(uint32_t rows, uint32_t per) { return ascq::walk_fits(rows, per); }\n'
                   'uint32_t columns(uint32_t j, uint32_t n) { return ascq::whole_columns(j, n); }\n'
                   'void shape(uint32_t lanes, uint32_t rows, uint32_t per, uint32_t* out)\n'
                   '{ auto w = ascq::row_walk(lanes, rows, per, 256); out[0] = w.grid_x; out[1] = w.grid_y; out[2] = w.block; }\n'
                   '}\n')
    lib = str(where / "t.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-o", lib, "-I",
                           os.path.join(ROOT, "asc-devkit_amd", "csrc"), str(src)])
    lib = C.CDLL(lib)
    lib.lanes.restype = lib.columns.restype = lib.fits.restype = C.c_uint32
    lib.lanes.argtypes, lib.columns.argtypes = [C.c_uint32], [C.c_uint32] * 2
    lib.fits.argtypes = [C.c_uint32] * 2
    lib.shape.argtypes = [C.c_uint32] * 3 + [C.POINTER(C.c_uint32)]
    return lib


@pytest.mark.parametrize("n", [8, 9, 15, 16, 2049, 2 ** 31 + 3, TOP - 9, TOP - 8, TOP - 7, TOP - 2, TOP - 1])
def test_every_column_has_a_lane(walk, n):
    lanes = -(-n // 8)
    assert walk.lanes(n) == lanes
    out = (C.c_uint32 * 3)()
    walk.shape(lanes, 1, 4, out)
    threads = out[0] * out[2]
    assert lanes <= threads < lanes + out[2] and out[1] == 1
    assert (threads - 1) * 8 < TOP                                      # a lane's first column fits 32 bits
    for lane in {0, lanes // 2, max(lanes - 2, 0), lanes - 1}:
        assert walk.columns(8 * lane, n) == min(8 * lane, n - 8)        # the last lane's columns end with the row
    for lane in range(lanes, min(threads, lanes + 64)):
        assert walk.columns(8 * lane, n) >= n                           # idle


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 65535 * 8, 2 ** 31, TOP - 8, TOP - 7, TOP - 1])
def test_every_row_count_has_groups(walk, rows):
    out = (C.c_uint32 * 3)()
    walk.shape(2, rows, 8, out)
    assert 1 <= out[1] <= min(65535, -(-rows // 8))
    # a workgroup's walk: the first row past the end fits 32 bits, or the rows are refused
    groups = out[1]
    past = [8 * y + -(-(rows - 8 * y) // (8 * groups)) * 8 * groups for y in {0, groups // 2, groups - 1}]
    assert not walk.fits(rows, 8) or max(past) < TOP
    assert walk.fits(rows, 8) == (rows <= TOP - 1 - 65535 * 8)


CHILD = """
import ctypes as C
from ascq import _abi as abi
L = abi.load_library()
d = abi.QuantDesc(policy=abi.PER_TENSOR, src_dtype=abi.BF16, compute=abi.COMPUTE_F32, round_mode=abi.CAST_RINT, k_dim=1, cal_count=%d)
print("status", L.ascq_quant(C.byref(d), C.c_void_p(1 << 44), C.c_void_p(1 << 20), None, None, None))
"""


@pytest.mark.parametrize("count", [TOP - 9, TOP - 7, TOP - 1])
def test_tensors_of_the_longest_odd_lengths_reach_their_launch(count):
    """No device is visible, so the launch itself fails and is reported; the way there must not end the process."""
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=os.path.join(ROOT, "asc-devkit_amd"))
    r = subprocess.run([sys.executable, "-c", CHILD % count], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert "status %d" % abi.EHIP in r.stdout
