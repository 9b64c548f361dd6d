"""The SPD inverse shared by several workgroups per matrix (GPU only): panels of four 16-blocks and
their remainders (10 to 16 blocks), in-place and strided calls, batches on both sides of the rule,
the failing pivot's index in every panel, replays of a captured call.

Tolerance: as for one workgroup per matrix, M eps cond(A) with cond(A) < 10: 6e-13.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 6e-13


def _matrix(M, batch, seed):
    W = np.random.RandomState(seed).randn(batch, M, 4 * M)
    return W @ W.transpose(0, 2, 1) / M


def _call(L, M, batch, A, lda, out, ldo, logdet, info):
    need = L.query('gpx_spd_workspace', M, batch)
    work = torch.full((max(need, 1),), float('nan'), dtype=torch.float64, device='cuda')
    L.call('gpx_spd_inv_batched_ws', M, batch, L.P(A), lda, M * lda, L.P(out), ldo, M * ldo, L.P(logdet), L.P(info),
           L.P(work) if need else None, L.S())
    return need, work


@pytest.mark.parametrize('M', [145, 160, 161, 176, 177, 192, 193, 200, 208, 209, 224, 240, 241, 255, 256])
@pytest.mark.parametrize('how', ['plain', 'inplace', 'strided'])
def test_split_inverse(M, how):
    from geepee_amd import _lib as L
    L.require_device()
    print('spd split', M, how, flush=True)
    batch, ld_ = 3, M + 5 if how == 'strided' else M
    A = _matrix(M, batch, M)
    buf = torch.zeros(batch, M, ld_, dtype=torch.float64, device='cuda')
    buf[:, :, :M] = torch.as_tensor(A, device='cuda')
    out = buf if how == 'inplace' else torch.full_like(buf, 7.0)
    logdet = torch.empty(batch, dtype=torch.float64, device='cuda')
    info = torch.full((batch,), -1, dtype=torch.int32, device='cuda')
    need, _ = _call(L, M, batch, buf, ld_, out, ld_, logdet, info)
    assert need > 0 and info.cpu().tolist() == [0] * batch
    ref = np.linalg.slogdet(A)[1]
    assert np.max(np.abs(logdet.cpu().numpy() - ref) / np.maximum(np.abs(ref), M)) < TOL
    X, R = out.cpu().numpy(), np.linalg.inv(A)
    assert (X[:, :, M:] == (7.0 if how == 'strided' else 0.0)).all()
    for b in range(batch):
        assert np.linalg.norm(X[b, :, :M] - R[b]) < TOL * np.linalg.norm(R[b])


@pytest.mark.parametrize('M,bad', [(160, 1), (200, 64), (200, 65), (200, 200), (256, 130), (256, 193), (256, 256)])
def test_split_first_bad_pivot(M, bad):
    from geepee_amd import _lib as L
    L.require_device()
    print('spd split bad pivot', M, bad, flush=True)
    A = _matrix(M, 2, M)
    A[1, bad - 1, bad - 1] = -100.0     # the leading minors before it stay positive definite
    t = torch.as_tensor(A, device='cuda')
    out, logdet = torch.empty_like(t), torch.empty(2, dtype=torch.float64, device='cuda')
    info = torch.empty(2, dtype=torch.int32, device='cuda')
    _call(L, M, 2, t, M, out, M, logdet, info)
    assert info.cpu().tolist() == [0, bad]
    assert torch.isnan(out[1]).all() and torch.isnan(logdet[1])
    assert torch.isfinite(out[0]).all() and torch.isfinite(logdet[0])


def test_split_rule_and_capture():
    from geepee_amd import _lib as L, dops
    L.require_device()
    size = lambda M, b: L.query('gpx_spd_workspace', M, b)
    assert size(128, 1) == size(144, 1) == size(256, 64) == size(300, 1) == size(256, 0) == size(0, 1) == 0
    assert size(160, 4) > 0 and size(160, 16) == 0 and size(256, 16) > 0
    A = torch.as_tensor(_matrix(200, 2, 5), device='cuda')
    want = dops.spd_inv(A)[0].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = dops.spd_inv(A)[0]
    for _ in range(3):
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize('M', [160, 177, 200, 256])
@pytest.mark.parametrize('ridge', [1e-3, 1e-6])
def test_split_matches_one_workgroup_ill_conditioned(M, ridge):
    """Both forms do the same operations tile for tile, so on matrices of condition 1e6 and 1e9 they
    give the same bits; their error against extended precision is within 4 cond eps."""
    from geepee_amd import _lib as L
    L.require_device()
    print('spd ill-conditioned', M, ridge, flush=True)
    rs = np.random.RandomState(M)
    X = rs.randn(2, M, M // 2)
    A = X @ X.transpose(0, 2, 1) + ridge * np.eye(M)
    t = torch.as_tensor(A, device='cuda')
    res = []
    for split in (True, False):
        out, ld = torch.empty_like(t), torch.empty(2, dtype=torch.float64, device='cuda')
        info = torch.empty(2, dtype=torch.int32, device='cuda')
        if split:
            assert _call(L, M, 2, t, M, out, M, ld, info)[0] > 0
        else:
            L.call('gpx_spd_inv_batched', M, 2, L.P(t), M, M * M, L.P(out), M, M * M, L.P(ld), L.P(info), L.S())
        assert info.cpu().tolist() == [0, 0]
        res.append((out, ld))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    for b in range(2):
        w = np.linalg.eigvalsh(A[b])
        R = np.linalg.inv(A[b]).astype(np.longdouble)
        Al = A[b].astype(np.longdouble)
        for _ in range(4):      # Newton steps in extended precision
            R = R @ (2 * np.eye(M) - Al @ R)
        err = np.linalg.norm((res[0][0][b].cpu().numpy() - R).astype(np.float64)) / np.linalg.norm(R.astype(np.float64))
        assert err < 4 * (w[-1] / w[0]) * 2.0 ** -52, err
