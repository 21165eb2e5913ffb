"""Bands, spline segments and placed templates of ``TemplateInterpFD`` from the device
kernels against torch's searchsorted and slices on the host, at the edges of their
tiles and of the grids. Whole numbers and copies: equal."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M,L,N", [(1, 1, 3, 1), (2, 6, 100, 1023), (3, 2, 257, 1024), (5, 3, 64, 4097),
                                     (300, 1, 4, 50)])
def test_bands_segments_and_fill(B, M, L, N, backend):
    import torch

    from bbhx_amd.waveformbuild import TemplateInterpFD

    rng = np.random.default_rng(B * N)
    f = np.sort(rng.uniform(0.0, 1.0, N))
    x = np.sort(rng.uniform(0.0, 1.0, (B, M, L)), axis=-1)
    x[:, :, 0] = f[rng.integers(0, N, (B, M))]  # knots on bins
    x = np.sort(x, axis=-1)
    x[0] += 0.25          # partly above the data
    if B > 1:
        x[1] = x[1] + 2.0  # wholly: an empty band
    if B > 2:
        x[2, 0, 1] = np.nan
    ft, xt = torch.as_tensor(f), torch.as_tensor(x)
    it = TemplateInterpFD(force_backend=backend)
    st, lengths, inds = it.band_indices(ft.cuda(), xt.cuda())
    want_st = torch.searchsorted(ft, xt.amin(dim=(1, 2)), right=True).numpy()
    want_et = torch.searchsorted(ft, xt.amax(dim=(1, 2)), right=True).numpy()
    assert st.dtype == np.int32 and lengths.dtype == np.int32
    assert np.array_equal(st, want_st) and np.array_equal(lengths, want_et - want_st)
    for b in range(B):
        vals = ft[st[b]:st[b] + lengths[b]][None].expand(M, -1).contiguous()
        want = torch.searchsorted(xt[b].contiguous(), vals, right=True) - 1
        assert inds[b].is_contiguous() and torch.equal(inds[b].cpu().reshape(M, -1).long(), want)
    n = int(lengths.sum())
    it.num_bin_all = B
    it._template_flat = torch.complex(torch.arange(3.0 * max(n, 1), dtype=torch.float64), torch.ones(1, dtype=torch.float64)).cuda()
    out = it.filled(N).cpu()
    flat, off = it._template_flat.cpu(), 0
    for b in range(B):
        want = torch.zeros((3, N), dtype=torch.complex128)
        want[:, st[b]:st[b] + lengths[b]] = flat[off:off + 3 * lengths[b]].reshape(3, -1)
        off += 3 * int(lengths[b])
        assert torch.equal(out[b], want)
