"""Looks through the machine code of kernels whose matrix instructions are written in inline assembly.

usage: check_matrix_asm.py a.o b.o ...   (exit status 1 when a wait is missing)

The compiler inserts the waits that a matrix instruction's result and operands need, but not for one in inline
assembly: to it the result is there at once, and it may place a copy, a conversion or a spill right behind the
instruction.  For every such instruction, on every path that follows it, this program wants
  * no instruction that reads or writes its result within kResult wait states (an instruction is one, s_nop n is
    n + 1), but for matrix instructions that accumulate in the same registers, and
  * no vector instruction that writes one of its operands within kOperand wait states before it.
In the kernels of COUNTED a step loads one operand into LDS and the other into registers, and its counted waits rest on both:
between two barriers either both kinds of loads are issued or none (the compiler drops a register load that nobody uses).
In the kernels of STAGED a stage's loads into LDS go out in one run, those into registers behind them, and the counted wait ahead of
a stage's LDS reads leaves the next stage's loads on their way: on every path to such a wait, its count is at most the
number of loads from the start of the last run on.  (Their matrix instructions are the compiler's own: it knows what they need.)
"""
import os
import re
import shutil
import subprocess
import sys
import tempfile

LLVM = os.environ.get("LLVM_BIN", "/opt/rocm/llvm/bin")
MATRIX = ("v_mfma_i32_16x16x64_i8", "v_mfma_f32_16x16x32_f16", "v_mfma_scale_f32_16x16x128_f8f6f4")
kResult, kOperand = 19, 2
COUNTED = ("wq_gemm_kernel",)
STAGED = ("wq_rows_kernel",)


def registers(operand):
    """'v[4:7]' -> {('v', 4), ...}; operands that are no vector registers -> empty"""
    m = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return frozenset()
    lo = int(m[2] if m[2] is not None else m[3])
    hi = int(m[2] if m[2] is not None else m[4])
    return frozenset((m[1], r) for r in range(lo, hi + 1))


class Instruction:
    def __init__(self, text, address):
        name, _, rest = text.partition(" ")
        self.text, self.name, self.address = text, name, address
        ops = [o.strip().split(" ")[0] for o in rest.split(",")] if rest else []
        self.ops = [registers(o) for o in ops]
        self.all = frozenset().union(*self.ops) if self.ops else frozenset()
        self.matrix = name in MATRIX
        store = name.startswith(("ds_write", "global_store", "buffer_store", "scratch_store", "v_cmp", "s_"))
        self.dst = frozenset() if store or not self.ops else self.ops[0]
        self.states = int(rest.split()[0]) + 1 if name == "s_nop" else 1
        self.target = None


def kernels(path):
    with tempfile.TemporaryDirectory() as tmp:
        copy = shutil.copy(path, tmp)
        subprocess.run([LLVM + "/llvm-objdump", "--offloading", copy], check=True, stdout=subprocess.DEVNULL)
        code = [f for f in os.listdir(tmp) if "amdgcn" in f]
        text = subprocess.run([LLVM + "/llvm-objdump", "-d", "--no-show-raw-insn", os.path.join(tmp, code[0])], check=True,
                              capture_output=True, text=True).stdout
    name, body = None, []
    for line in text.splitlines():
        m = re.match(r"([0-9a-f]+) <(\S+)>:$", line)
        if m:
            if body:
                yield name, body
            name, body, start = m[2], [], int(m[1], 16)
            continue
        m = re.match(r"\s+([a-z]\w*(?: .*?)?)\s*// ([0-9A-F]+):(?: <\S+?\+0x([0-9a-f]+)>)?", line)
        if m and name:
            i = Instruction(m[1].strip(), int(m[2], 16))
            if i.name.startswith(("s_cbranch", "s_branch")):
                t = re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>\s*$", line)
                if not t:
                    raise SystemExit("check_matrix_asm: no target in %r" % line)
                i.target = start + int(t[1] or "0", 16)
            body.append(i)
    if body:
        yield name, body


def faults(body):
    where = {i.address: n for n, i in enumerate(body)}

    def follow(n, budget, visit, seen):
        """visit(instruction) -> True: this path is settled; every path from n on for `budget` wait states"""
        while budget > 0 and n < len(body):
            if seen.get(n, 0) >= budget:
                return
            seen[n] = budget
            i = body[n]
            if visit(i):
                return
            budget -= i.states
            if i.name in ("s_endpgm", "s_setpc_b64"):
                return
            if i.target is not None:
                follow(where[i.target], budget, visit, seen)
                if i.name == "s_branch":
                    return
            n += 1

    bad = []
    for n, m in enumerate(body):
        if m.matrix:
            result = m.ops[0]

            def used(i):
                if i.all & result:
                    if not (i.matrix and i.ops[0] == result and i.ops[3] == result and not (i.ops[1] | i.ops[2]) & result):
                        bad.append("%s  before the result of  %s" % (i.text, m.text))
                    return True
                return False
            follow(n + 1, kResult, used, {})
        elif m.dst and m.name.startswith("v_"):
            def fed(i):
                if i.matrix and i.all & m.dst:
                    bad.append("%s  reads what  %s  wrote just before" % (i.text, m.text))
                return False
            follow(n + 1, kOperand, fed, {})
    return bad


def dropped_loads(body):
    bad, lds, reg = [], 0, 0
    for i in body:
        if i.name.startswith(("global_load_lds", "buffer_load")) or i.name.startswith("global_load"):
            if "_lds" in i.name or i.text.endswith(" lds"):
                lds += 1
            else:
                reg += 1
        elif i.name == "s_barrier":
            if lds and not reg:
                bad.append("%d loads into LDS and none into registers before the barrier at %x" % (lds, i.address))
            lds = reg = 0
    return bad


def loose_waits(body):
    where = {i.address: n for n, i in enumerate(body)}

    def guards(n):
        """the count of a wait with LDS reads behind it (no other access or matrix instruction in between)"""
        m = re.search(r"vmcnt\((\d+)\)", body[n].text) if body[n].name == "s_waitcnt" else None
        for i in body[n + 1:] if m else ():
            if i.name.startswith("ds_read"):
                return int(m[1])
            if i.name.startswith(("ds_", "buffer_", "global_", "v_mfma", "s_waitcnt", "s_barrier", "s_branch", "s_cbranch", "s_endpgm")):
                break
        return None

    bad, seen, work = [], set(), [(0, 0, False)]               # instruction, loads since the last run's start, still in the run
    while work:
        n, loads, run = work.pop()
        while n < len(body) and (n, loads, run) not in seen:
            seen.add((n, loads, run))
            i = body[n]
            if i.name.startswith(("buffer_load", "global_load")):
                lds = "_lds" in i.name or i.text.endswith(" lds")
                loads, run = (1 if lds and not run else min(loads + 1, 64)), lds
            left = guards(n)
            if left is not None and left > loads:
                bad.append("%s at %x leaves more than the %d loads since the last run into LDS began" % (i.text, i.address, loads))
            if i.target is not None:
                work.append((where[i.target], loads, run))
                if i.name == "s_branch":
                    break
            if i.name in ("s_endpgm", "s_setpc_b64"):
                break
            n += 1
    return sorted(set(bad))


def main(paths):
    status = 0
    for path in paths:
        seen = 0
        for name, body in kernels(path):
            count = sum(i.matrix for i in body)
            seen += count
            staged = any(c in name for c in STAGED)
            bad = loose_waits(body) if staged else faults(body) if count else []
            if any(c in name for c in COUNTED):
                bad += dropped_loads(body)
            for b in bad[:10]:
                sys.stderr.write("check_matrix_asm: %s: %s\n" % (name, b))
            status |= bool(bad)
        if not seen:
            sys.stderr.write("check_matrix_asm: no matrix instruction found in %s\n" % path)
            status = 1
    return status


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
