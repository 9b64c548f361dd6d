"""The SPD inverse at the edges of its storage layouts (GPU only): tiles of 16 rows, the sizes
where the matrix moves from registers to LDS and to the output array, in-place and
log-determinant-only calls, row strides larger than M, and the failing pivot's index.

Tolerance: a backward-stable inverse has relative error of order M eps cond(A); the matrices
are W W^T / M with W of M x 4M Gaussians, condition number below 10 (Marchenko-Pastur edge
((1 + 1/2) / (1 - 1/2))^2 = 9), so 256 * 2.2e-16 * 10 = 6e-13 bounds it; the log-determinant, a
sum of M terms of order one, gets the same bound.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 6e-13


def _matrix(M, batch, seed):
    rs = np.random.RandomState(seed)
    W = rs.randn(batch, M, 4 * M)
    return W @ W.transpose(0, 2, 1) / M


@pytest.mark.parametrize('M', [1, 15, 16, 17, 48, 49, 144, 145, 192, 193, 208, 209, 224, 225, 240, 241, 255, 256])
@pytest.mark.parametrize('how', ['plain', 'inplace', 'strided', 'logdet'])
def test_spd_layouts(M, how):
    from geepee_amd import _lib as L
    L.require_device()
    print('spd', M, how, flush=True)
    batch = 3
    A = _matrix(M, batch, M)
    ld_ = M + 5 if how == 'strided' else M
    buf = torch.zeros(batch, M, ld_, dtype=torch.float64, device='cuda')
    buf[:, :, :M] = torch.as_tensor(A, device='cuda')
    out = None if how == 'logdet' else (buf if how == 'inplace' else torch.full_like(buf, 7.0))
    logdet = torch.empty(batch, dtype=torch.float64, device='cuda')
    info = torch.full((batch,), -1, dtype=torch.int32, device='cuda')
    L.call('gpx_spd_inv_batched', M, batch, L.P(buf), ld_, M * ld_, L.P(out), ld_, M * ld_, L.P(logdet),
           L.P(info), L.S())
    assert info.cpu().tolist() == [0] * batch
    ref = np.linalg.slogdet(A)[1]
    assert np.max(np.abs(logdet.cpu().numpy() - ref) / np.maximum(np.abs(ref), M)) < TOL
    if out is not None:
        X = out.cpu().numpy()
        assert (X[:, :, M:] == (7.0 if how == 'strided' else 0.0)).all()
        R = np.linalg.inv(A)
        for b in range(batch):
            assert np.linalg.norm(X[b, :, :M] - R[b]) < TOL * np.linalg.norm(R[b])


@pytest.mark.parametrize('M,bad', [(16, 1), (50, 17), (130, 130), (200, 64), (256, 3), (256, 241)])
def test_spd_first_bad_pivot(M, bad):
    from geepee_amd import _lib as L
    L.require_device()
    print('spd bad pivot', M, bad, flush=True)
    A = _matrix(M, 2, M)
    A[1, bad - 1, bad - 1] = -100.0     # the leading minors before it stay positive definite
    t = torch.as_tensor(A, device='cuda')
    out, logdet = torch.empty_like(t), torch.empty(2, dtype=torch.float64, device='cuda')
    info = torch.empty(2, dtype=torch.int32, device='cuda')
    L.spd_inv(t, out, logdet, info)
    assert info.cpu().tolist() == [0, bad]
    assert torch.isnan(out[1]).all() and torch.isnan(logdet[1])
    assert torch.isfinite(out[0]).all() and torch.isfinite(logdet[0])
