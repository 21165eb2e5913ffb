"""The device kernel of the A, E and T noise PSDs against the host formulas, at the
edges of its launch and of the frequency range.

Tolerance: the host takes 1 - cos x by subtraction, which loses up to 2^-53 of 1, so
S_T there is off by up to 2e-16 / (1 - cos x) of itself; 1e-14 for the rest (some
twenty roundings, and sin x of x up to 6 near its zero at pi, relative to the largest
phase's rounding: 1e-15 / |sin x|).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 70001])
def test_aet1_psd_matches_host(n, backend):
    import torch

    from bbhx_amd.utils.constants import C_SI
    from bbhx_amd.utils.sensitivity import LISA_L, AET1SensitivityMatrix

    f = np.logspace(-6, -1, n)
    f_d = torch.as_tensor(f, device="cuda")
    sens, host = AET1SensitivityMatrix(f[:1]), AET1SensitivityMatrix(f)
    psd = sens.update_frequency_tensor(f_d, f, backend)
    assert psd.shape == (3, n) and np.array_equal(sens.frequency_arr, f)
    x = 2 * np.pi * LISA_L / C_SI * f
    tol = 1e-14 + 4 * 1e-15 / np.abs(np.sin(x))
    for i in range(3):
        assert np.array_equal(psd[i].cpu().numpy(), sens[i])
        rel = np.abs(sens[i] / host[i] - 1)
        bound = tol + (2.3e-16 / (1 - np.cos(x)) if i == 2 else 0.0)
        print(n, i, rel.max(), np.max(rel / bound), flush=True)
        assert np.all(rel <= bound)
