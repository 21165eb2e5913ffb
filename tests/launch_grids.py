"""Launches that the library makes for given sizes, recorded on a host without a
GPU (launch_recorder.cpp takes the place of the HIP runtime). Run in a process of
its own, ``python launch_grids.py recorder.so case``; prints the launches as JSON."""

import ctypes as C
import json
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT))


class Library:
    def __init__(self, recorder):
        self.rec = C.CDLL(recorder, mode=C.RTLD_GLOBAL)
        self.rec.recorder_kernel.restype = C.c_char_p
        self.rec.recorder_arg.restype = C.c_int64
        from bbhx_amd.cutils import load_library

        self.lib = load_library()
        self.launches = []

    def call(self, name, *args, args_of="-", nargs=0):
        """Status of an entry point; its launches as (kernel, grid, block, args)."""
        self.rec.recorder_clear(args_of.encode(), nargs)
        status = getattr(self.lib, "bbhx_hip_" + name)(*args)
        self.launches = []
        for i in range(self.rec.recorder_count()):
            g = (C.c_uint64 * 6)()
            self.rec.recorder_grid(i, g)
            kernel = self.rec.recorder_kernel(i).decode()
            a = [self.rec.recorder_arg(i, k) for k in range(nargs)] if args_of in kernel else []
            self.launches.append((kernel, list(g[:3]), list(g[3:]), a))
        return status


def interpolate(lib, n, params, sets):
    p = [C.c_void_p(4096)] * 6
    return lib.call("interpolate", *p, n, params, 1, sets, None, args_of="k_spline", nargs=12)


CASES = {"interpolate": interpolate}


if __name__ == "__main__":
    lib = Library(sys.argv[1])
    out = []
    for name, *args in json.loads(sys.argv[2]):
        status = CASES[name](lib, *args)
        out.append(dict(status=status, launches=lib.launches))
    print(json.dumps(out))
