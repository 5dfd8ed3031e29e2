"""The build's look through the machine code of matrix instructions in inline assembly, on a few lines of code."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "asc-devkit_amd", "csrc"))
import check_matrix_asm as check  # noqa: E402

MFMA = "v_mfma_i32_16x16x64_i8 v[0:3], v[8:11], v[12:15], v[0:3]"
OTHER = "v_mfma_i32_16x16x64_i8 v[4:7], v[8:11], v[12:15], v[4:7]"


def body(*lines):
    """instructions at addresses 0, 4, ...; 'L: s_branch' forms jump to the line whose number follows '->'"""
    out = []
    for n, line in enumerate(lines):
        text, _, target = line.partition(" -> ")
        i = check.Instruction(text, 4 * n)
        i.target = 4 * int(target) if target else None
        out.append(i)
    return out


@pytest.mark.parametrize("lines,wrong", [
    ((MFMA, OTHER, MFMA, "s_nop 15", "s_nop 15", "v_cvt_f32_i32_e32 v20, v0", "s_endpgm"), False),
    ((MFMA, OTHER, "s_nop 7", "v_cvt_f32_i32_e32 v20, v2", "s_endpgm"), True),                 # read too early
    ((MFMA, "v_mov_b32_e32 v3, v20", "s_endpgm"), True),                                       # overwritten
    ((MFMA, "global_store_dwordx4 v[20:21], v[0:3], off", "s_endpgm"), True),                  # stored too early
    ((MFMA, "v_mfma_i32_16x16x64_i8 v[4:7], v[0:3], v[12:15], v[4:7]", "s_endpgm"), True),     # an operand of the next one
    ((MFMA, "v_mfma_i32_16x16x64_i8 v[4:7], v[8:11], v[12:15], v[0:3]", "s_endpgm"), True),    # added up elsewhere
    (("v_cvt_f32_i32_e32 v20, v0", "s_nop 15", MFMA, "s_cbranch_scc1 s -> 0", "s_endpgm"), True),   # round the loop
    (("v_cvt_f32_i32_e32 v20, v0", "s_nop 15", MFMA, "s_nop 15", "s_nop 15", "s_cbranch_scc1 s -> 0", "s_endpgm"), False),
    (("v_mov_b32_e32 v9, v20", MFMA, "s_nop 15", "s_nop 15", "s_endpgm"), True),               # operand written just before
    (("v_mov_b32_e32 v9, v20", "s_nop 1", MFMA, "s_endpgm"), False),
    (("ds_read_b128 v[8:11], v30", "s_waitcnt lgkmcnt(0)", MFMA, "s_endpgm"), False),
])
def test_missing_waits_are_found(lines, wrong):
    assert bool(check.faults(body(*lines))) == wrong


def test_loads_that_the_compiler_dropped_are_found():
    """A counted wait of the half GEMM rests on a step's loads into LDS and into registers: a stretch between two barriers with
    the first kind alone means that the compiler has left the second out."""
    step = ["global_load_lds_dwordx4 v1, s[0:1]", "buffer_load_dwordx4 v[4:7], v2, s[4:7], 0 offen", "s_waitcnt vmcnt(6)", "s_barrier"]
    assert check.dropped_loads(body(*step, *step, *step[2:])) == []          # whole steps, and one that loads nothing
    assert len(check.dropped_loads(body(*step, *step[:1], *step[2:]))) == 1
    # (a buffer load into LDS counts as such)
    assert len(check.dropped_loads(body("buffer_load_dwordx4 v1, s[4:7], 0 offen lds", "s_barrier"))) == 1


def test_waits_that_count_more_loads_than_there_are_are_found():
    """The whole-k tiles: a stage is a run of loads into LDS and the loads into registers behind it; the wait ahead of a stage's LDS reads
    leaves the next stage on its way.  Too large a count, a load between those of the run, and both only on one path."""
    lds, reg, read = "buffer_load_dwordx4 v1, s[4:7], s9 offen lds", "buffer_load_dwordx2 v[4:5], v2, s[8:11], s9 offen", "ds_read_b128 v[8:11], v3"
    stage = [lds, lds, reg]

    def loop(count, prologue, steady=stage):
        start = len(prologue)
        step = ["s_waitcnt vmcnt(%d)" % count, read, *steady]
        return body(*prologue, *step, *step, "s_cbranch_scc1 s -> %d" % start, "s_waitcnt vmcnt(0)", "s_endpgm")
    assert check.loose_waits(loop(3, stage + stage)) == []
    assert check.loose_waits(loop(4, stage + stage))                               # a load that is counted and not issued
    assert check.loose_waits(loop(3, [lds, reg, lds] * 2))                         # the last of the run behind a register load
    assert check.loose_waits(loop(3, stage + [reg, lds, lds]))                     # the run behind the register loads
    assert check.loose_waits(loop(3, stage + stage, [lds, lds]))                   # a register load dropped from the steps
    assert check.loose_waits(body(*stage, "s_cbranch_scc1 s -> 5", reg, "s_nop 0", "s_waitcnt vmcnt(4)", read, "s_endpgm"))  # on one path
    assert check.loose_waits(body(*stage, *stage, "s_waitcnt vmcnt(9)", "v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[8:11], v[0:3]", "s_endpgm")) == []
