"""Short sparse grids share workgroups in the direct likelihood's splines and their
adjoint: a batch of mixed short and long grids against the kernel-by-kernel path,
whose splines are another kernel's, and beside a template that is not a number.

Tolerance: 1e-7 (|d_h| + h_h): the phases reach 1e6-1e7 rad, so a bin's term may
differ by ~1e-8 of itself between the two paths.
"""

import numpy as np
import pytest

from tests.params import MODES, YRSID_SI, draw, perturb
from tests.test_gpu_direct_grad import to_sampling

pytestmark = pytest.mark.gpu

LENGTHS = np.array([4, 16, 64, 128, 5, 300, 100, 129, 33, 4, 4, 127, 7, 64, 64, 16], dtype=np.int32)


def test_packed_splines_in_a_mixed_batch(backend):
    from bbhx_amd.likelihood import Likelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    wave = BBHWaveformFD(response_kwargs=dict(orbits=EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI), tdi2=True),
                         force_backend=backend)
    ref = draw(1, 1001)[:, 0]
    ref[0], ref[1], ref[11] = 1.3e6, 4.1e5, 0.62 * YRSID_SI
    f = np.arange(1, 8193) * (16.0 / YRSID_SI)
    sens = AET1SensitivityMatrix(f)
    data = wave(*ref, freqs=f, length=1024, modes=MODES, direct=False, fill=True)[0]
    like = Likelihood(wave, f, data, np.array([sens[0], sens[1], sens[2]]), force_backend=backend)
    p = perturb(ref, LENGTHS.size, 22, scale=1e-3)
    like.get_ll_fused(p, LENGTHS, modes=MODES)
    d_h, h_h = like.d_h.cpu().numpy(), like.h_h.cpu().numpy().real
    for b, length in enumerate(LENGTHS):
        like.get_ll(p[:, b:b + 1], length=int(length), modes=MODES)
        want_d, want_h = like.d_h.cpu().numpy()[0], like.h_h.cpu().numpy()[0].real
        tol = 1e-7 * (abs(want_d) + want_h)
        print(length, d_h[b], want_d, flush=True)
        assert abs(d_h[b] - want_d) <= tol and abs(h_h[b] - want_h) <= tol
    # a template that is not a number leaves the others as they are
    x = to_sampling(p)
    ll, grad = like.get_ll_and_grad_fused(x, LENGTHS, modes=MODES)
    bad = 9
    x[bad, 4] = np.nan
    ll_bad, grad_bad = like.get_ll_and_grad_fused(x, LENGTHS, modes=MODES)
    rest = np.arange(LENGTHS.size) != bad
    assert not np.isfinite(ll_bad[bad]) and np.isfinite(ll_bad[rest]).all()
    assert np.array_equal(ll[rest], ll_bad[rest])
    assert np.allclose(grad[rest], grad_bad[rest], rtol=1e-9, atol=1e-9 * np.abs(grad[rest]).max())
