"""Binaries' parameters given as columns (B, 1), which count as their B entries, as
they did when each was copied to the device by itself."""

import numpy as np
import pytest
import torch

from tests.params import MODES, YRSID_SI, draw


def test_rows_of_any_shape_in_one_copy():
    from bbhx_amd.utils.arrays import rows_to_dev

    rows = [np.arange(5.0), np.arange(3.0)[:, None], np.asfortranarray(np.arange(6.0).reshape(2, 3)), np.zeros(0)]
    out = rows_to_dev(rows, "cpu")
    for r, t in zip(rows, out):
        assert t.dtype == torch.float64 and np.array_equal(t.numpy(), r.flatten())


@pytest.mark.gpu
def test_columns_equal_rows(backend):
    from bbhx_amd.response.fastfdresponse import LISATDIResponse
    from bbhx_amd.utils.orbits import EqualArmlengthOrbits
    from bbhx_amd.waveforms.phenomhm import PhenomHMAmpPhase

    B, L = 3, 64
    p = draw(B, 7)
    wave = PhenomHMAmpPhase(force_backend=backend)
    resp = LISATDIResponse(orbits=EqualArmlengthOrbits(dt=1e4, t_max=3.0 * YRSID_SI), force_backend=backend)
    out = []
    for shape in (lambda v: v, lambda v: v[:, None]):
        m1, m2, c1, c2, dist, phi, f_ref, inc, lam, beta, psi = (shape(v) for v in p[:11])
        wave(m1, m2, c1, c2, dist, phi, f_ref, p[11], L, modes=MODES, Tobs=np.full(B, YRSID_SI))
        freqs, phase, tf = wave.freqs_shaped.clone(), wave.phase.clone(), wave.tf.clone()
        resp(freqs, inc, lam, beta, psi, phi, L, modes=MODES, phase=phase, tf=tf)
        out.append([freqs.cpu(), wave.amp.cpu(), phase.cpu(), resp.response_carrier.cpu()])
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)
    for bad in (p[11][:, None], p[11][:2], np.zeros(4)):
        with pytest.raises(ValueError, match="t_ref"):
            wave(*p[:7], bad, L, modes=MODES, Tobs=np.full(B, YRSID_SI))
