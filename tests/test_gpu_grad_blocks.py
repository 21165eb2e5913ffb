"""The heterodyned gradient at node counts around its workgroups (one lane per node,
256 nodes per workgroup) against central differences of the FP64 CPU oracle.

Compared are distance, phi_ref, cos inc and psi, which shift no node across the
observation window. Tolerance: 1e-7 (|d_h| + h_h) per component, the distance's times
the distance: both sides are FP64, the terms of the sums differ by up to ~1e-8 of
themselves (phases of 1e6-1e7 rad) and their derivatives by up to 4 times that; the
fourth-order quotient of d_h - h_h / 2 with steps of 1e-3 adds less.
"""

import numpy as np
import pytest

from oracle.pipeline import OracleHeterodyne, OracleWaveform
from tests.params import MODES, YRSID_SI, draw
from tests.test_gpu_adjoint_pass import COMPONENTS, STEP
from tests.test_gpu_grad import to_sampling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [16, 63, 65, 255, 256, 257, 600])
def test_grad_blocks_match_oracle_differences(K, backend):
    from bbhx_amd.likelihood import HeterodynedLikelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    orbits = EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI)
    ref = draw(1, 1001)[:, 0]
    ref[0], ref[1], ref[11] = 1.3e6, 4.1e5, 0.62 * YRSID_SI
    f = np.arange(1, 2**13 + 1) * (16.0 / YRSID_SI)
    owave = OracleWaveform(orbits.as_host_dict(), tdi2=True)
    data = owave(*ref, freqs=f, length=1024, modes=MODES, direct=False, fill=True, squeeze=True)[0]
    wave = BBHWaveformFD(response_kwargs=dict(orbits=orbits, tdi2=True), force_backend=backend)
    het = HeterodynedLikelihood(wave, f, data, ref, K, sens_mat=AET1SensitivityMatrix(f),
                                template_gen_kwargs=dict(modes=MODES),
                                reference_gen_kwargs=dict(length=1024, modes=MODES), force_backend=backend)
    psd_fn = lambda x: [AET1SensitivityMatrix(x)[i] for i in range(3)]  # noqa: E731
    ohet = OracleHeterodyne(owave, f, data, ref, K, psd_fn, reference_length=1024, modes=MODES)
    x0 = to_sampling(ref[:, None])[0]
    rng = np.random.default_rng(K)
    X = x0[None, :] + np.array([3e-6, 1e-4, 3e-4, 3e-4, 0.0, 0.05, 0.02, 0.001, 0.001, 0.05, 0.3]) * rng.standard_normal((2, 11))
    X[:, 4] = x0[4] * (1 + 0.01 * rng.standard_normal(2))
    _, grad = het.get_ll_and_grad(X)

    def oracle(Y):
        _, d_h, h_h = ohet.get_ll(HeterodynedLikelihood.sampling_to_params(Y))
        return np.real(d_h), np.real(h_h)

    d_h, h_h = oracle(X)
    scale = np.abs(d_h) + np.abs(h_h)
    assert np.all(np.isfinite(grad))
    for what, k in COMPONENTS.items():
        unit = X[:, k] if what == "dist" else np.ones(2)
        lls = []
        for s in (2, 1, -1, -2):
            Y = X.copy()
            Y[:, k] += s * STEP * unit
            d, h = oracle(Y)
            lls.append(d - 0.5 * h)
        fd = (-lls[0] + 8 * lls[1] - 8 * lls[2] + lls[3]) / (12 * STEP)
        err = np.abs(grad[:, k] * unit - fd)
        print(K, what, grad[:, k] * unit, "error", err, "scale", scale, flush=True)
        assert np.all(err <= 1e-7 * scale)
