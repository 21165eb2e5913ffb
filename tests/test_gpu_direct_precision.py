"""``precision`` of the direct likelihood: 1 (log-likelihoods within 1e-3 suffice) is
evaluated as 0 is, in FP64, and equals it bit for bit; other values are refused."""

import numpy as np
import pytest

from tests.params import MODES, YRSID_SI, draw

pytestmark = pytest.mark.gpu


def test_precision_one_equals_zero(backend):
    from bbhx_amd.cutils import HipCallError
    from bbhx_amd.likelihood import Likelihood
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.utils.sensitivity import AET1SensitivityMatrix
    from bbhx_amd.waveformbuild import BBHWaveformFD

    wave = BBHWaveformFD(response_kwargs=dict(orbits=EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI), tdi2=True),
                         force_backend=backend)
    p = draw(5, 1003)
    lengths = np.array([64, 300, 512, 777, 128], dtype=np.int32)
    f = np.arange(1, 8193) * (16.0 / YRSID_SI)
    sens = AET1SensitivityMatrix(f)
    data = wave(*p[:, 0], freqs=f, length=1024, modes=MODES, direct=False, fill=True)[0]
    like = Likelihood(wave, f, data, np.array([sens[0], sens[1], sens[2]]), force_backend=backend)
    plan = like.direct_plan(lengths, MODES)
    size = plan.nbytes()
    out = []
    for precision in (0, 1, 0):
        ll = like.get_ll_fused(p, lengths, modes=MODES, plan=plan, precision=precision)
        out.append([ll, like.d_h.cpu().numpy(), like.h_h.cpu().numpy()])
    for other in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], other))
    assert plan.nbytes() == size
    for bad in (2, -1):
        with pytest.raises(HipCallError):
            plan.set_precision(bad)
    assert plan.precision == 0
