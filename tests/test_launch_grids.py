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


def spline_blocks(n):
    return 1 if n <= 256 else 1 + -(-(n - 256) // 160)


@pytest.mark.parametrize("groups,modes", [([(5, 64), (1, 4096), (3, 100)], 6), ([(1, 4), (2, 257)], 1),
                                          ([(40, 300), (2, 129)], 3), ([(70, 4), (3, 128), (9, 5)], 6)])
def test_direct_work_by_length(record, groups, modes):
    """An uneven batch's launches hold the workgroups of its grids' own lengths and no others."""
    cases = [("direct", groups, modes, 4096, *k) for k in
             (("k_dir_spline", 3, 4), ("k_dirg_spline_adj", 3, 4, True), ("k_dirg_knots", 4, 4, True))]
    spline, adj, knots = record(*cases)
    lengths = [length for n, length in groups for _ in range(n)]
    for r, kernel in ((spline, "k_dir_spline"), (adj, "k_dirg_spline_adj")):
        want = [(b * modes + m, k) for b, n in enumerate(lengths) if n > 128 for m in range(modes)
                for k in range(spline_blocks(n))]
        blocks = len(want)
        rows, got = r["rows"], []
        assert sum(g[0] for g, _, _ in launches(r, kernel)) == len(rows)
        for first, sets, lanes, block in rows[:blocks]:
            assert (sets, lanes) == (1, 256)
            got.append((first, block))
        want += [(b * modes + m, 0) for b, n in enumerate(lengths) if n <= 128 for m in range(modes)]
        for first, sets, lanes, block in rows[blocks:]:
            assert sets * lanes <= 256 and block == 0
            assert lanes == max(lengths[(first + k) // modes] for k in range(sets))
            got += [(first + k, 0) for k in range(sets)]
        assert got == want
    work = modes * sum(n * -(-length // 256) for n, length in groups)
    assert sum(g[0] for g, _, _ in launches(knots, "k_dirg_knots")) == work
    assert knots["table"]["size"] == knots["table"]["distinct"] == work
    assert knots["table"]["high"][2] == work - 1
    grid = {}
    for n, length in groups:
        lanes = 64 if length <= 64 else 128 if length <= 128 else 256
        grid[lanes] = grid.get(lanes, 0) + n * modes
    assert {b[0]: g[0] for g, b, _ in launches(spline, "k_dir_grid")} == grid


def test_short_direct_grids_share_workgroups(record):
    r, = record(("direct", [(1000, 16)], 6, 1024, "k_dir_spline", 3, 4))
    assert [g[0] for g, _, _ in launches(r, "k_dir_spline")] == [6000 // 16]


def test_direct_grids_of_many_templates(record):
    """More (template, mode) pairs than one launch of 256 lanes each holds."""
    n = 2_900_000
    forward, = record(("direct", [(n, 129)], 6, 1024, "k_dir_spline", 3, 4))
    assert sum(g[0] for g, _, _ in launches(forward, "k_dir_grid")) == 6 * n
    assert forward["table"] == dict(size=6 * n, distinct=6 * n, low=[0, 1, 256, 0], high=[6 * n - 1, 1, 256, 0])
    grad, = record(("direct", [(n, 193)], 6, 1024, "k_dirg_knots", 4, 4, True))
    assert sum(g[0] for g, _, _ in launches(grad, "k_dirg_knots")) == 6 * n
    assert grad["table"]["distinct"] == 6 * n and grad["table"]["high"][2] == 6 * n - 1


@pytest.mark.parametrize("grad", [False, True])
def test_heterodyned_wavefronts(record, grad):
    """One wavefront per 64 nodes where the modes of the last nodes are not spread over others, or
    where four have nodes already."""
    sizes = [(16, 300, 6, 5), (16, 320, 1, 5), (16, 128, 6, 8), (16, 64, 6, 1), (16, 1000, 6, 8), (300, 448, 6, 7),
             (16, 192, 6, 8), (16, 193, 6, 4), (16, 256, 6, 4)]
    for (batch, nodes, modes, waves), r in zip(sizes, record(*[("heterodyned", *s[:3], grad) for s in sizes])):
        (grid, block, _), = launches(r, "k_grad_weights" if grad else "k_fused_eval")
        assert (grid[0], block[0]) == (batch, 64 * waves)


@pytest.mark.parametrize("batch,nodes,modes", [(3_000_000, 256, 6), (2_800_000, 300, 6), (17_000_000, 65, 1),
                                               (100, 300, 6)])
def test_heterodyned_gradient_of_many_templates(record, batch, nodes, modes):
    """Every (template, mode)'s chunks of nodes are launched, whatever their number."""
    r, = record(("heterodyned", batch, nodes, modes, True))
    done = {}
    for grid, block, args in launches(r, "k_grad_points"):
        row0, node0, chunk0, chunks = (a & 0xFFFFFFFF for a in args[15:19])
        rows, lanes = done.get((node0, chunk0, chunks), (0, block[0]))
        assert row0 == rows and grid[0] % chunks == 0 and lanes == block[0]
        done[node0, chunk0, chunks] = rows + grid[0] // chunks, lanes
    node = chunk = 0
    for (node0, chunk0, chunks), (rows, lanes) in done.items():
        assert (node0, chunk0, rows) == (node, chunk, batch * modes)
        node, chunk = node0 + chunks * lanes, chunk0 + chunks
    assert nodes <= node < nodes + 256 and chunk == -(-nodes // 256)


def test_template_grids_of_many_binaries(record):
    """Bands, segments and placement of batches beyond one launch: every binary's workgroups,
    its arrays where they were."""
    base = 1 << 20
    bands, segments, fill = record(("interp_bands", 20_000_000, 2, 4), ("interp_segments", 1900, 6, 1_580_000),
                                   ("fill_bands", 600, 12_600_000))
    done = 0
    for grid, _, args in launches(bands, "k_interp_bands"):
        assert args[0] == base + 8 * done and args[1] == base + 8 * done * 2 * 4
        done += grid[0]
    assert done == 20_000_000
    done, tiles = 0, -(-1_580_000 // 1024)
    for grid, _, args in launches(segments, "k_interp_segments"):
        assert args[8] & 0xFFFFFFFF == done and grid[0] % tiles == 0
        done += grid[0] // tiles
    assert done == 1900 * 6
    done, tiles = 0, -(-12_600_000 // 256)
    for grid, _, args in launches(fill, "k_fill_bands"):
        assert args[0] == base + 16 * 3 * 12_600_000 * done and args[1] == base
        assert args[2] == base + 8 * done and args[3] == base + 8 * done
        done += grid[0] // tiles
    assert done == 600


def test_waveform_grids_of_many_points(record):
    """The waveform's frequency grids and time shift beyond one launch of a lane per point."""
    batch, modes, length = 3_000_000, 6, 300
    points = batch * modes * length
    for what, kernel, at in (("phm_default_grid", "k_phm_default_grid", 8), ("phm_time_shift", "k_phm_time_shift", 6)):
        r, = record((what, batch, modes, length))
        done = 0
        for grid, _, args in launches(r, kernel):
            assert args[at:at + 2] == [256 * done, points]
            done += grid[0]
        assert done == -(-points // 256)
    r, = record(("phm_refit_grid", batch, modes, length))
    done = 0
    for grid, _, args in launches(r, "k_phm_refit_grid"):
        assert args[9] & 0xFFFFFFFF == done
        done += grid[0]
    assert done == batch * modes


def test_noise_of_many_frequencies(record):
    n = 5_000_000_000
    r, = record(("aet1_psd", n))
    done = 0
    for grid, _, args in launches(r, "k_aet1_psd"):
        assert args[2] == n and args[6] == 256 * done
        done += grid[0]
    assert done == -(-n // 256)
