"""Which kernels a call launches, found without a GPU: a child process loads the library behind tests/cpp/launch_log.cpp, which
writes launches down instead of running them.  A route is what the host code chooses for 256 compute units (what the library
assumes where it cannot ask a device)."""
import ctypes as C
import functools
import json
import os
import subprocess
import sys
from typing import NamedTuple

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOG = os.path.join(ROOT, "tests", "cpp", "launch_log.so")


class Launch(NamedTuple):
    kernel: str        # name with its template arguments, without namespaces
    grid_x: int
    grid_y: int
    block: int

    @property
    def name(self):
        return self.kernel.split("<")[0]

    @property
    def args(self):
        """the template arguments as text"""
        return tuple(a.strip() for a in self.kernel.partition("<")[2].rstrip(">").split(","))


def routes(calls):
    """calls: [(entry point, [argument, ...])], an argument being a number, None, or (descriptor class name, {field: value}).
    Returns [(status, [Launch, ...])]."""
    assert os.path.exists(LOG), "tests/cpp/launch_log.so is not built: run __graft_entry__.build()"
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=os.path.join(ROOT, "asc-devkit_amd"))
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], input=json.dumps(calls), env=env, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return [(status, [Launch(n, int(x), int(y), int(b)) for n, x, y, b in launches]) for status, launches in json.loads(r.stdout)]


def route(entry, *args):
    """the kernels of one call that is accepted"""
    return _route(entry, json.dumps(args))


@functools.lru_cache(maxsize=None)
def _route(entry, args):
    (status, launches), = routes([(entry, json.loads(args))])
    assert status == 0, (entry, args, status)
    return launches


def _child():
    from ascq import _abi as abi
    log = C.CDLL(LOG, mode=C.RTLD_GLOBAL)
    log.launch_log_take.restype = C.c_char_p
    lib = C.CDLL(abi.LIB_PATH)
    out = []
    for entry, args in json.load(sys.stdin):
        fn = getattr(lib, entry)
        fn.restype, fn.argtypes = abi.SIGNATURES[entry]
        held = [getattr(abi, a[0])(**a[1]) if isinstance(a, list) else a for a in args]
        status = fn(*[C.byref(h) if isinstance(h, C.Structure) else h for h in held])
        lines = log.launch_log_take().decode().splitlines()
        out.append((status, [line.rsplit(";", 3) for line in lines]))
    json.dump(out, sys.stdout)


if __name__ == "__main__":
    _child()
