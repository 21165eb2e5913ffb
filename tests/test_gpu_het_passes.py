"""The heterodyned likelihood where the last pass over the nodes spreads its modes over
the lanes of a wavefront or the wavefronts of a template, and around those sizes,
against the FP64 CPU oracle.

Tolerance: |delta logL| <= 1e-6 + 1e-8 (|d_h| + h_h): both sides are FP64 and the phases,
of 1e6-1e7 rad, move each term of the sums by up to ~1e-8 of itself.
"""

import numpy as np
import pytest

from oracle.pipeline import OracleHeterodyne, OracleWaveform
from tests.params import MODES, YRSID_SI, draw, perturb

pytestmark = pytest.mark.gpu


# 3 templates: up to eight wavefronts each; 300: seven, 700: three; 2100: one
@pytest.mark.parametrize("modes", [MODES, [(3, 3)], MODES[:3]], ids=["6", "1", "3"])
@pytest.mark.parametrize("K", [8, 32, 33, 65, 96, 97, 128, 200, 257, 768])
def test_het_passes_match_oracle(K, modes, backend):
    from bbhx_amd.likelihood import HeterodynedLikelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    orbits = EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI)
    ref = draw(1, 1001)[:, 0]
    ref[0], ref[1], ref[11] = 1.3e6, 4.1e5, 0.62 * YRSID_SI
    f = np.arange(1, 2**13 + 1) * (16.0 / YRSID_SI)
    owave = OracleWaveform(orbits.as_host_dict(), tdi2=True)
    data = owave(*ref, freqs=f, length=1024, modes=modes, direct=False, fill=True, squeeze=True)[0]
    wave = BBHWaveformFD(response_kwargs=dict(orbits=orbits, tdi2=True), force_backend=backend)
    het = HeterodynedLikelihood(wave, f, data, ref, K, sens_mat=AET1SensitivityMatrix(f),
                                template_gen_kwargs=dict(modes=modes),
                                reference_gen_kwargs=dict(length=1024, modes=modes), force_backend=backend)
    psd_fn = lambda x: [AET1SensitivityMatrix(x)[i] for i in range(3)]  # noqa: E731
    ohet = OracleHeterodyne(owave, f, data, ref, K, psd_fn, reference_length=1024, modes=modes)
    p = perturb(ref, 3, 22, scale=1e-5)
    want, d_h, h_h = ohet.get_ll(p)
    bound = 1e-6 + 1e-8 * (np.abs(d_h) + np.abs(h_h))
    for B in (3, 300, 700, 2100):
        print(K, len(modes), B, flush=True)
        ll = het.get_ll(np.tile(p, (1, B // 3)), fused=True).reshape(-1, 3)
        assert np.array_equal(ll, np.tile(ll[:1], (B // 3, 1)))
        print(np.abs(ll[0] - want), bound, flush=True)
        assert np.all(np.abs(ll[0] - want) <= bound)
