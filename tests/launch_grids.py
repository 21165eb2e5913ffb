"""Launches that the library makes for given sizes, recorded on a host without a
GPU (launch_recorder.cpp takes the place of the HIP runtime). Run in a process of
its own, ``python launch_grids.py recorder.so case``; prints the launches as JSON."""

import ctypes as C
import json
import sys
from pathlib import Path

import numpy as np

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
        if not self.rec.recorder_count():
            return status
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


def ints(v):
    return np.ascontiguousarray(v, dtype=np.int32).ctypes.data_as(C.POINTER(C.c_int))


def mode_list(modes):
    return np.array([(2, 2), (2, 1), (3, 3), (3, 2), (4, 4), (4, 3)][:modes], dtype=np.int32).T.copy()


def response(lib):
    resp, p = C.c_void_p(), C.c_void_p(4096)
    links = ints([12, 23, 31, 13, 32, 21])
    assert lib.call("response_create", C.byref(resp)) == 0
    assert lib.call("response_add_orbits", resp, 1e4, 100, p, p, p, links, links, links, 2.5e9) == 0
    return resp


def heterodyned(lib, batch, nodes, modes, grad=False):
    p, lm, resp = C.c_void_p(4096), mode_list(modes), response(lib)
    args = [*([p] * (6 if grad else 5)), batch, ints(lm[0]), ints(lm[1]), modes, p, p, p, nodes, p, 1001, 2e-3, 0.0,
            resp, 0, 0, 1, 0]
    if grad:
        return lib.call("hdyn_fused_grad", *args, p, 0.0, None, args_of="k_grad_points", nargs=19)
    return lib.call("hdyn_fused", *args, 0, p, 0.0, None)


def direct(lib, groups, modes, bins, kernel, table, width, grad=False):
    """A direct call on templates of (count, length) groups; also the entries of the work
    table that argument ``table`` of the kernel's launches points to, ``width`` ints each."""
    p = C.c_void_p(4096)
    lengths = np.concatenate([np.full(n, length, dtype=np.int32) for n, length in groups])
    resp, plan = response(lib), C.c_void_p()
    status = lib.call("direct_plan_create", C.byref(plan), len(lengths), ints(lengths), modes, bins, 1024)
    if status == 0 and grad:
        status = lib.call("direct_plan_enable_grad", plan)
    if status:
        return status
    lm = mode_list(modes)
    out = [p] * (4 if grad else 3)
    status = lib.call("direct_fused_grad" if grad else "direct_fused", plan, *out, p, p, p, ints(lm[0]), ints(lm[1]),
                      modes, p, p, p, p, 1001, 2e-3, 0.0, 1e-4, 0.6, resp, 0, 0, 1, 16384, 256, 2048, None,
                      args_of=kernel, nargs=table + 1)
    rows = []
    for k, grid, _, args in lib.launches:
        if kernel in k:
            buf = (C.c_int * (width * grid[0])).from_address(args[table])
            rows.append(np.frombuffer(buf, dtype=np.int32).reshape(-1, width))
    lib.extra = summary(np.concatenate(rows)) if rows else None
    lib.call("direct_plan_destroy", plan)
    return status


def summary(table):
    """A table's size, how many of its rows differ in the first two entries, and their range."""
    key = table[:, 0].astype(np.int64) << 32 | table[:, 1]
    out = dict(size=len(table), distinct=len(np.unique(key)), low=table.min(0).tolist(), high=table.max(0).tolist())
    return dict(table=out, rows=table.tolist() if len(table) < 10000 else None)


P = C.c_void_p(1 << 20)
CALLS = {
    "interp_bands": lambda lib, batch, modes, length: lib.call(
        "interp_bands", P, P, P, P, length, 1000, batch, modes, None, args_of="k_interp_bands", nargs=5),
    "interp_segments": lambda lib, batch, modes, longest: lib.call(
        "interp_segments", P, P, P, P, P, 64, longest, batch, modes, None, args_of="k_interp_segments", nargs=9),
    "fill_bands": lambda lib, batch, bins: lib.call(
        "fill_bands", P, P, P, P, bins, batch, None, args_of="k_fill_bands", nargs=6),
    "phm_default_grid": lambda lib, batch, modes, length: lib.call(
        "phm_default_grid", P, P, P, P, -4.0, -0.2, length, modes, batch, None, args_of="grid", nargs=10),
    "phm_time_shift": lambda lib, batch, modes, length: lib.call(
        "phm_time_shift", P, P, P, 0.0, length, modes, batch, None, args_of="shift", nargs=8),
    "phm_refit_grid": lambda lib, batch, modes, length: lib.call(
        "phm_refit_grid", P, P, P, P, None, 1, 0, length, modes, batch, None, args_of="refit", nargs=10),
    "aet1_psd": lambda lib, n: lib.call(
        "aet1_psd", P, P, n, 2.5e9, 3e-15, 1.5e-11, None, args_of="k_aet1_psd", nargs=7),
}
CASES = {"interpolate": interpolate, "direct": direct, "heterodyned": heterodyned, **CALLS}


if __name__ == "__main__":
    lib = Library(sys.argv[1])
    out = []
    for name, *args in json.loads(sys.argv[2]):
        lib.launches, lib.extra = [], None
        status = CASES[name](lib, *args)
        out.append(dict(status=status, launches=lib.launches, **(lib.extra or {})))
    print(json.dumps(out))
