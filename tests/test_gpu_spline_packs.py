"""Short sets of knots share a workgroup of the batched splines: each of them against
scipy's not-a-knot spline, and a set that holds a NaN beside the others.

Tolerance as for the longer ones (test_gpu_spline_blocks.py): 1e-11 of the system's
largest |y| for slopes and coefficients in units of the segment's width.
"""

import numpy as np
import pytest
from scipy.interpolate import CubicSpline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,P,sets", [(4, 9, 64), (4, 1, 131), (5, 3, 103), (16, 2, 17), (63, 4, 9), (64, 9, 5),
                                      (100, 3, 3), (127, 1, 5), (128, 9, 3), (129, 3, 3)])
def test_short_sets_match_scipy(L, P, sets, backend):
    import torch

    from bbhx_amd.utils.interpolate import CubicSplineInterpolant

    rng = np.random.default_rng(L)
    x = np.cumsum(rng.uniform(0.2, 2.0, (sets, 1, L)), axis=-1)
    y = rng.standard_normal((P, sets, 1, L))
    bad = sets // 2
    y[:, bad, 0, L // 2] = np.nan
    spl = CubicSplineInterpolant(torch.as_tensor(x, device="cuda"), torch.as_tensor(y, device="cuda"),
                                 force_backend=backend)
    c1, c2, c3, slope = (c.cpu().numpy().reshape(P, sets, L) for c in (spl.c1, spl.c2, spl.c3, spl.B))
    for p in range(P):
        for b in range(sets):
            if b == bad:
                assert not np.isfinite(c1[p, b]).all()
                continue
            cs = CubicSpline(x[b, 0], y[p, b, 0], bc_type="not-a-knot")
            scale, h = np.abs(y[p, b, 0]).max(), np.diff(x[b, 0])
            for got, want in ((c1[p, b, :-1] * h, cs.c[2] * h), (c2[p, b, :-1] * h**2, cs.c[1] * h**2),
                              (c3[p, b, :-1] * h**3, cs.c[0] * h**3), (slope[p, b, 1:] * h, cs(x[b, 0, 1:], 1) * h)):
                assert np.max(np.abs(got - want)) <= 1e-11 * scale, (p, b)
            assert c1[p, b, -1] == c2[p, b, -1] == c3[p, b, -1] == 0.0
