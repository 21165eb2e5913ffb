"""The heterodyned gradient of a batch large enough for a launch of its own for the
nodes that fill no workgroup, against the same templates in a batch of two (whose
gradients test_gpu_grad_blocks.py holds against the oracle).

Tolerance: 1e-9 of the batch's largest component: the sums are taken in another order,
and their terms exceed them by less than 10^5, so 1e-16 of the terms is 1e-11.
"""

import numpy as np
import pytest

from tests.params import MODES, YRSID_SI, draw
from tests.test_gpu_grad import to_sampling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,B", [(257, 683), (257, 682), (320, 700), (448, 683), (449, 683), (513, 342)])
def test_grad_of_a_large_batch(K, B, backend):
    from bbhx_amd.likelihood import HeterodynedLikelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    ref = draw(1, 1001)[:, 0]
    ref[0], ref[1], ref[11] = 1.3e6, 4.1e5, 0.62 * YRSID_SI
    f = np.arange(1, 2**13 + 1) * (16.0 / YRSID_SI)
    wave = BBHWaveformFD(response_kwargs=dict(orbits=EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI), tdi2=True),
                         force_backend=backend)
    data = wave(*ref, freqs=f, length=1024, modes=MODES, direct=False, fill=True)[0]
    het = HeterodynedLikelihood(wave, f, data, ref, K, sens_mat=AET1SensitivityMatrix(f),
                                template_gen_kwargs=dict(modes=MODES),
                                reference_gen_kwargs=dict(length=1024, modes=MODES), force_backend=backend)
    x0 = to_sampling(ref[:, None])[0]
    rng = np.random.default_rng(K)
    X = x0 + np.array([3e-6, 1e-4, 3e-4, 3e-4, 0.0, 0.05, 0.02, 0.001, 0.001, 0.05, 0.3]) * rng.standard_normal((B, 11))
    ll, grad = het.get_ll_and_grad(X)
    assert np.isfinite(grad).all()
    pick = [0, B - 1]
    ll2, grad2 = het.get_ll_and_grad(X[pick])
    scale = np.abs(grad).max(axis=0)
    print(K, B, (np.abs(grad[pick] - grad2) / scale).max(), flush=True)
    assert np.all(np.abs(grad[pick] - grad2) <= 1e-9 * scale)
