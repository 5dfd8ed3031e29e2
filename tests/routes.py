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


class Calls:
    """The child process; it ends with this one."""

    def __init__(self):
        assert os.path.exists(LOG), "tests/cpp/launch_log.so is not built: run __graft_entry__.build()"
        env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=os.path.join(ROOT, "asc-devkit_amd"))
        self.child = subprocess.Popen([sys.executable, os.path.abspath(__file__)], env=env, stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)

    def __call__(self, entry, args):
        self.child.stdin.write(json.dumps([entry, args]) + "\n")
        self.child.stdin.flush()
        status, lines = json.loads(self.child.stdout.readline())
        return status, [Launch(n, int(x), int(y), int(b)) for n, x, y, b in lines]


@functools.lru_cache(maxsize=None)
def _calls():
    return Calls()


def call(entry, *args):
    """(status, [Launch, ...]) of one call; an argument is a number, None, or (descriptor class name, {field: value}), fields likewise."""
    return _calls()(entry, args)


def route(entry, *args):
    """The kernels of one call that is accepted."""
    status, launches = call(entry, *args)
    assert status == 0, (entry, args, status)
    return launches


def _child():
    from ascq import _abi as abi

    def held(a):
        return getattr(abi, a[0])(**{field: held(v) for field, v in a[1].items()}) if isinstance(a, list) else a

    log = C.CDLL(LOG, mode=C.RTLD_GLOBAL)
    log.launch_log_take.restype = C.c_char_p
    lib = C.CDLL(abi.LIB_PATH)
    for line in sys.stdin:
        entry, args = json.loads(line)
        fn = getattr(lib, entry)
        fn.restype, fn.argtypes = abi.SIGNATURES[entry]
        status = fn(*[C.byref(h) if isinstance(h, C.Structure) else h for h in map(held, args)])
        print(json.dumps([status, [text.rsplit(";", 3) for text in log.launch_log_take().decode().splitlines()]]), flush=True)


if __name__ == "__main__":
    _child()
