"""The batched spline solver at the edges of its blocks of knots and groups of
quantities against scipy's not-a-knot spline.

Tolerance: 1e-11 of the system's largest |y|, for the slopes and coefficients in units
of the segment's width (slope h, c2 h^2, c3 h^3). The systems are diagonally dominant
by two, so the solutions carry a few tens of roundings of the right sides, which
neighbouring spacings (their ratio below 10 here) enlarge by up to 10^2: 1e-13.
"""

import numpy as np
import pytest
from scipy.interpolate import CubicSpline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,P,B,M", [(3, 1, 2, 1), (4, 2, 3, 1), (5, 9, 1, 2), (64, 4, 2, 2), (255, 3, 1, 1),
                                     (256, 9, 2, 1), (257, 5, 1, 3), (416, 1, 3, 1), (417, 9, 1, 1), (577, 2, 1, 1),
                                     (8096, 9, 1, 6)])
def test_spline_blocks_match_scipy(L, P, B, M, backend):
    import torch

    from bbhx_amd.utils.interpolate import CubicSplineInterpolant

    rng = np.random.default_rng(L)
    x = np.cumsum(rng.uniform(0.2, 2.0, (B, M, L)) * np.logspace(0, 3, L), axis=-1)
    y = np.sin(np.linspace(0, 0.3 * L, L) * (1 + 0.1 * np.arange(P)[:, None, None, None])) + rng.standard_normal(
        (P, B, M, L))
    spl = CubicSplineInterpolant(torch.as_tensor(x, device="cuda"), torch.as_tensor(y, device="cuda"),
                                 force_backend=backend)
    c1, c2, c3 = (c.cpu().numpy().reshape(P, B, M, L) for c in (spl.c1, spl.c2, spl.c3))
    slope = spl.B.cpu().numpy().reshape(P, B, M, L)
    h = np.diff(x, axis=-1)
    worst = 0.0
    for p in range(P):
        for b in range(B):
            for m in range(M):
                cs = CubicSpline(x[b, m], y[p, b, m], bc_type="not-a-knot")
                scale = np.abs(y[p, b, m]).max()
                hb = h[b, m]
                for got, want in ((c1[p, b, m, :-1] * hb, cs.c[2] * hb), (c2[p, b, m, :-1] * hb**2, cs.c[1] * hb**2),
                                  (c3[p, b, m, :-1] * hb**3, cs.c[0] * hb**3),
                                  (slope[p, b, m, 1:] * hb, cs(x[b, m, 1:], 1) * hb)):
                    err = np.max(np.abs(got - want)) / scale
                    worst = max(worst, err)
                    assert err <= 1e-11, (p, b, m)
                assert c1[p, b, m, -1] == c2[p, b, m, -1] == c3[p, b, m, -1] == 0.0
    print(L, P, "worst", worst, flush=True)
