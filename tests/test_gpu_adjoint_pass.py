"""The adjoint dense pass and the adjoint of the splines of the direct likelihood's
gradient at the sizes where their blocks, work items and segment search have edges,
against central differences of the FP64 CPU oracle, template by template.

Compared are the components that leave the sparse grid and the observation window
where they are (distance, phi_ref, cos inc, psi); the gradient holds those two fixed.

Tolerance: 1e-7 (|d_h| + h_h) per component, the distance's times the distance. The
phases reach 1e6-1e7 rad, so a bin's term differs by up to ~1e-8 of itself between the
two and its derivative by up to 4 (the highest m) times that; the fourth-order
quotient with steps of 1e-3 adds 1e-12 / 1e-3 of rounding and (4e-3)^4 / 30 of
truncation, both relative to the same scale.
"""

import numpy as np
import pytest

from oracle.pipeline import OracleLikelihood, OracleWaveform
from tests.params import MODES, YRSID_SI, draw, perturb
from tests.test_gpu_direct_grad import to_sampling

pytestmark = pytest.mark.gpu

COMPONENTS = {"dist": 4, "phi": 5, "cosi": 6, "psi": 9}
STEP = 1e-3

# bins, spacing, sparse lengths, (chunk, min_chunk, block), (t_obs_start, t_obs_end), modes
CASES = {
    "40_bins": (40, "uniform", [300, 4], (16384, 1024, 256), (0.0, 1.0), MODES),
    "257_bins": (257, "uniform", [300, 64], (64, 64, 128), (0.0, 1.0), MODES),
    "short_grids": (5001, "uniform", [4, 5, 7, 33], (16384, 1024, 256), (0.0, 1.0), MODES),
    "long_grids": (1501, "uniform", [3000], (4096, 1024, 256), (0.0, 1.0), MODES),
    "spline_blocks": (1001, "uniform", [6, 255, 256, 257, 258, 415, 417, 577], (16384, 1024, 256), (0.0, 1.0), MODES),
    "odd_chunk": (3001, "uniform", [500, 256], (1000, 1000, 256), (0.0, 1.0), MODES),
    "log_spaced": (2000, "log", [700, 256], (16384, 1024, 256), (0.0, 1.0), MODES),
    "window": (5001, "uniform", [16, 300], (16384, 1024, 256), (0.05, 0.5), MODES),
    "one_mode": (5001, "uniform", [64, 300], (16384, 1024, 256), (0.0, 1.0), [(3, 3)]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_adjoint_pass_matches_oracle_differences(name, backend):
    from bbhx_amd.likelihood import HeterodynedLikelihood, Likelihood
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
    X = to_sampling(perturb(ref, lengths.size, 22, scale=1e-2))
    plan = like.direct_plan(lengths, modes, chunk=chunk, block=block, min_chunk=min_chunk)
    print(name, lengths, flush=True)
    _, grad = like.get_ll_and_grad_fused(X, lengths, modes=modes, plan=plan, t_obs_start=t0, t_obs_end=t1)

    def oracle(x, b):
        p = HeterodynedLikelihood.sampling_to_params(x[None, :])
        _, d_h, h_h = olike.get_ll(p, length=int(lengths[b]), modes=modes, t_obs_start=t0, t_obs_end=t1)
        return d_h[0], h_h[0]

    for b in range(lengths.size):
        d_h, h_h = oracle(X[b], b)
        scale = abs(d_h) + abs(h_h)
        assert np.all(np.isfinite(grad[b]))
        for what, k in COMPONENTS.items():
            unit = X[b, k] if what == "dist" else 1.0
            lls = []
            for s in (2, 1, -1, -2):
                y = X[b].copy()
                y[k] += s * STEP * unit
                d_h, h_h = oracle(y, b)
                lls.append(np.real(d_h) - 0.5 * np.real(h_h))  # without <d|d>, which the quotient would have to cancel
            fd = (-lls[0] + 8 * lls[1] - 8 * lls[2] + lls[3]) / (12 * STEP)
            err = abs(grad[b, k] * unit - fd)
            print(name, lengths[b], what, grad[b, k] * unit, "error", err, "scale", scale, flush=True)
            assert err <= 1e-7 * scale
