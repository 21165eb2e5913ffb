"""Grids of the library's launches at sizes no GPU test reaches (CPU: the launches
are recorded, not made). HIP takes fewer than 2^32 work-items per grid dimension."""

import json
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
LIB = ROOT / "bbhx_amd" / "libbbhx_hip.so"
HERE = Path(__file__).resolve().parent

pytestmark = pytest.mark.skipif(not LIB.exists(), reason="libbbhx_hip.so not built")


@pytest.fixture(scope="module")
def record(tmp_path_factory):
    so = tmp_path_factory.mktemp("recorder") / "recorder.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(so), str(HERE / "launch_recorder.cpp")], check=True)

    def run(*cases):
        out = subprocess.run([sys.executable, str(HERE / "launch_grids.py"), str(so), json.dumps(cases)],
                             capture_output=True, text=True, check=True, timeout=300)
        return json.loads(out.stdout)

    return run


def launches(result, kernel):
    """The (grid, block, args) of one kernel; every launch of the call within HIP's limit."""
    assert result["status"] == 0
    for _, grid, block, _ in result["launches"]:
        assert all(0 < g * b < 2**32 for g, b in zip(grid, block)), (grid, block)
    return [(g, b, a) for k, g, b, a in result["launches"] if kernel in k]


def test_spline_grids(record):
    """Every (set of knots, group of quantities) has its workgroups, whatever the number of
    sets; short sets share them."""
    sizes = [(300, 9, 4_000_000), (129, 9, 6_000_000), (128, 9, 6_000_001), (4, 9, 6_000_000), (3, 1, 40_000_000),
             (1 << 28, 2, 3)]
    for (n, params, sets), r in zip(sizes, record(*[("interpolate", *s) for s in sizes])):
        blocks = 1 if n <= 256 else 1 + -(-(n - 256) // 160)
        done = 0
        for grid, block, args in launches(r, "k_spline"):
            assert args[11] & 0xFFFFFFFF == done and grid[0] % blocks == 0
            done += grid[0] // blocks
        packs = -(-sets // (256 // n)) if n <= 128 else sets
        assert done == packs * (-(-params // 3) if params >= 3 else params)
