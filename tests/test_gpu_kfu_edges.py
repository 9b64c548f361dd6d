"""The SE kernel matrix and its adjoint at the edges of their thread layouts (GPU only): columns
per block (64, 128, 256), row batches of four, register widths (Q = 4, 8, 12, 16) and the
general path beyond 16 inputs.

Tolerance: r^2/2 of magnitude E < 200 carries an absolute error of a few E eps into the
exponential (< 2e-13 relative); the adjoint's sums of up to 20000 terms of mixed sign lose at
most two digits more: 1e-11 normwise.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _nrel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize('N,M,Q', [(1, 1, 1), (15, 63, 4), (16, 64, 5), (17, 65, 8), (100, 128, 9), (33, 129, 12),
                                   (64, 256, 13), (2049, 200, 16), (20001, 40, 3), (5, 70, 17), (40, 9, 30)])
def test_se_and_adjoint(N, M, Q):
    from geepee_amd import dops
    print('se', N, M, Q, flush=True)
    rs = np.random.RandomState(N + M + Q)
    x, z, ls, sf = rs.randn(N, Q), rs.randn(M, Q), 0.2 * rs.randn(Q) + 0.5, np.array([0.3])
    G = rs.randn(N, M)
    t = [torch.as_tensor(a, device='cuda') for a in (x, z, ls, sf, G)]
    il = np.exp(-2 * ls)
    K = np.exp(2 * sf[0] - 0.5 * (((x * np.sqrt(il)) ** 2).sum(1)[:, None] + ((z * np.sqrt(il)) ** 2).sum(1)[None]
                                  - 2 * (x * il).dot(z.T)))
    got = dops.se(t[0], t[1], t[2], t[3])
    assert _nrel(got.cpu().numpy(), K) < 1e-11
    if N == 1 or M < 2:
        return
    Kzz = dops.se(t[1], t[1], t[2], t[3], jitter=0.25).cpu().numpy()
    assert np.array_equal(Kzz, Kzz.T) and np.allclose(np.diag(Kzz), np.exp(2 * sf[0]) + 0.25, rtol=1e-14)
    if Q > 16:
        return
    L = G * K
    dsf2, dell, dz, dx = dops.kfu_bwd(t[4], got, t[0], t[1], t[2], t[3], want_dx=True)
    cs = L.sum(0)
    assert abs(float(dsf2) - L.sum() / np.exp(2 * sf[0])) < 1e-11 * np.abs(L).sum() / np.exp(2 * sf[0])
    wl = np.array([(L * (z[None, :, q] - x[:, q:q + 1]) ** 2).sum() for q in range(Q)]) * np.exp(-3 * ls)
    assert _nrel(dell.cpu().numpy(), wl) < 1e-10
    assert _nrel(dz.cpu().numpy(), -(z * cs[:, None] - L.T.dot(x)) * il) < 1e-11
    assert _nrel(dx.cpu().numpy(), (L.dot(z) - x * L.sum(1)[:, None]) * il) < 1e-11


@pytest.mark.parametrize('Q', [3, 8, 16])
@pytest.mark.parametrize('N,M', [(1536, 64), (1537, 64), (3072, 64), (3073, 64), (4096, 64), (4097, 64), (2049, 65),
                                 (3073, 32), (8193, 31), (6145, 16), (16385, 15), (70, 17), (70, 33)])
def test_se_rows_per_block(N, M, Q):
    """Entries are the same bits from one and from four rows a thread and from 16, 32 and 64 columns a
    block (on both sides of each line)."""
    from geepee_amd import dops
    print('se rows', N, M, Q, flush=True)
    rs = np.random.RandomState(N + Q)
    x, z, ls, sf = [torch.as_tensor(a, device='cuda') for a in (rs.randn(N, Q), rs.randn(M, Q), 0.2 * rs.randn(Q),
                                                                 np.array([0.3]))]
    K = dops.se(x, z, ls, sf)
    for r0, r1 in ((0, 1), (3, 40), (N - 17, N)):
        assert torch.equal(K[r0:r1], dops.se(x[r0:r1].contiguous(), z, ls, sf))
    c = min(M, 16)
    assert torch.equal(K[:, :c], dops.se(x, z[:c].contiguous(), ls, sf))


@pytest.mark.parametrize('N,M,Q', [(960, 30, 5), (961, 30, 5), (480, 100, 3), (481, 100, 9), (240, 200, 16), (241, 200, 2)])
def test_kfu_rows_per_thread(N, M, Q):
    """The adjoint on both sides of 60 blocks of four rows a thread, against two halves of the rows
    (1e-12 of the sums' terms, of either sign: 1e-11 normwise)."""
    from geepee_amd import dops
    print('kfu rows', N, M, Q, flush=True)
    rs = np.random.RandomState(N + Q)
    x, z, ls, sf, G = [torch.as_tensor(a, device='cuda') for a in (rs.randn(N, Q), rs.randn(M, Q), 0.2 * rs.randn(Q) + 0.5,
                                                                    np.array([0.3]), rs.rand(N, M))]
    K = dops.se(x, z, ls, sf)
    whole = dops.kfu_bwd(G, K, x, z, ls, sf, want_dx=True)
    cut = [[t[a:b].contiguous() for t in (G, K, x)] for a, b in ((0, N // 2), (N // 2, N))]
    parts = [dops.kfu_bwd(g, k, xx, z, ls, sf, want_dx=True) for g, k, xx in cut]
    for i in range(3):
        assert _nrel(whole[i].cpu().numpy(), (parts[0][i] + parts[1][i]).cpu().numpy()) < 1e-11
    assert torch.equal(whole[3], torch.cat([p[3] for p in parts]))
