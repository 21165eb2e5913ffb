"""The dense pass and the splines of the fused direct likelihood at the sizes where
their blocks, work items and segment search have edges, against the FP64 CPU oracle run
template by template.

Tolerance: |delta logL| <= 1e-6 + 1e-8 (|d_h| + h_h). Both sides are FP64; the
phases reach 1e6-1e7 rad, so one rounding of a phase is 1e-9 rad and a few of
them move each bin's term by up to ~1e-8 of itself.
"""

import numpy as np
import pytest

from oracle.pipeline import OracleLikelihood, OracleWaveform
from tests.params import MODES, YRSID_SI, draw, perturb

pytestmark = pytest.mark.gpu

# bins, spacing, sparse lengths, (chunk, min_chunk, block), (t_obs_start, t_obs_end), modes
CASES = {
    # fewer bins than a wavefront; one block, one more, one less
    "40_bins": (40, "uniform", [300, 4], (16384, 1024, 256), (0.0, 1.0), MODES),
    "255_bins": (255, "uniform", [300, 64], (64, 64, 64), (0.0, 1.0), MODES),
    "257_bins": (257, "uniform", [300, 64], (64, 64, 128), (0.0, 1.0), MODES),
    # segments of thousands of bins, and several segments to a bin
    "short_grids": (20001, "uniform", [4, 5, 7, 33], (16384, 1024, 256), (0.0, 1.0), MODES),
    "long_grids": (3001, "uniform", [4096, 3000], (4096, 1024, 256), (0.0, 1.0), MODES),
    # the spline's row blocks of 256 knots, one more every 160
    "spline_blocks": (2001, "uniform", [6, 255, 256, 257, 258, 415, 416, 417, 576, 577], (16384, 1024, 256), (0.0, 1.0),
                      MODES),
    # items that are not a multiple of a block, the last one short
    "odd_chunk": (9001, "uniform", [500, 256], (1000, 1000, 256), (0.0, 1.0), MODES),
    # uneven data frequencies; blocks that start below the grid and end above it
    "log_spaced": (5000, "log", [700, 256], (16384, 1024, 256), (0.0, 1.0), MODES),
    # an observation window that cuts the segments of every mode, and one mode
    "window": (20001, "uniform", [16, 300], (16384, 1024, 256), (0.05, 0.5), MODES),
    "one_mode": (20001, "uniform", [64, 300], (16384, 1024, 256), (0.0, 1.0), [(3, 3)]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_dense_pass_matches_oracle(name, backend):
    from bbhx_amd.likelihood import Likelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    n, spacing, lengths, (chunk, min_chunk, block), (t0, t1), modes = CASES[name]
    orbits = EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI)
    ref = draw(1, 1001)[:, 0]
    ref[0], ref[1], ref[11] = 1.3e6, 4.1e5, 0.62 * YRSID_SI
    f = 1e-5 + np.arange(n) * (4e-3 / n) if spacing == "uniform" else np.logspace(-5, -1.5, n)
    owave = OracleWaveform(orbits.as_host_dict(), tdi2=True)
    inj = owave(*ref, freqs=f, length=512, modes=MODES, direct=False, fill=True, squeeze=True)[0]
    sens = AET1SensitivityMatrix(f)
    psd = np.array([sens[0], sens[1], sens[2]])
    like = Likelihood(BBHWaveformFD(response_kwargs=dict(orbits=orbits, tdi2=True), force_backend=backend), f, inj, psd,
                      force_backend=backend)
    olike = OracleLikelihood(owave, f, inj, psd)
    lengths = np.asarray(lengths, dtype=np.int32)
    p = perturb(ref, lengths.size, 22, scale=1e-5)
    plan = like.direct_plan(lengths, modes, chunk=chunk, block=block, min_chunk=min_chunk)
    print(name, lengths, flush=True)
    ll = like.get_ll_fused(p, lengths, modes=modes, plan=plan, t_obs_start=t0, t_obs_end=t1)
    for b, length in enumerate(lengths):
        want, d_h, h_h = olike.get_ll(p[:, b:b + 1], length=int(length), modes=modes, t_obs_start=t0, t_obs_end=t1)
        err, scale = abs(ll[b] - want[0]), abs(d_h[0]) + abs(h_h[0])
        print(name, length, "logL", ll[b], "error", err, "scale", scale, flush=True)
        assert np.isfinite(ll[b])
        assert err <= 1e-6 + 1e-8 * scale
