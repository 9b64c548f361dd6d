"""The q(u) chain's fused launches at their edges (GPU only): outer products and a second output in
a product's epilogue (every kernel a product can take), means and second moments, the
hyper-parameter tail, the KL term.

Tolerance: sums of at most 5000 products of order one in a different order than numpy's: 1e-12
normwise (the KL's scalar: relative to the sum of magnitudes).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _nrel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device='cuda')


# rank-1, matrix-vector, 16 x 16, 32 x 32 (one wave and four per tile), split K, and a size
# that without a tail takes 64 x 64 tiles
@pytest.mark.parametrize('b,m,n,k,splits', [(1, 9, 11, 1, 1), (3, 20, 1, 7, 1), (1, 50, 50, 50, 1), (2, 17, 33, 40, 1),
                                            (60, 100, 100, 40, 1), (70, 128, 130, 20, 1), (1, 30, 40, 2000, 4),
                                            (2, 0, 5, 3, 1), (40, 300, 300, 64, 1)])
def test_product_tail(b, m, n, k, splits):
    from geepee_amd import _lib as L
    print('tail', b, m, n, k, splits, flush=True)
    rs = np.random.RandomState(b + m + n + k)
    A, B, E, E2, C0 = rs.randn(b, m, k), rs.randn(b, k, n), rs.randn(m, n), rs.randn(b, m, n), rs.randn(b, m, n)
    U, V = rs.randn(b, m), rs.randn(b, n)
    R = 0.7 * A @ B + E
    S = R - 1.5 * U[:, :, None] * V[:, None, :]
    C, C2 = _dev(C0), _dev(np.zeros((b, m, n)))
    args = dict(alpha=0.7, E=_dev(E), gamma=1.0, splits=splits)
    L.mm(_dev(A), _dev(B), C, outer=(_dev(U), _dev(V), -1.5), **args)
    assert _nrel(C.cpu().numpy(), S) < 1e-12
    L.mm(_dev(A), _dev(B), C, outer=(_dev(U), _dev(V), -1.5), second=(C2, 0.3, _dev(E2)), **args)
    assert _nrel(C.cpu().numpy(), R) < 1e-12 and _nrel(C2.cpu().numpy(), 0.3 * S + E2) < 1e-12
    L.mm(_dev(A), _dev(B), C, second=(C2, 2.0, None), beta=0.5, **args)
    assert _nrel(C2.cpu().numpy(), 2.0 * (1.5 * R)) < 1e-12
    # several outer products into one matrix
    C = _dev(C0[0])
    L.mm(_dev(A[0]), _dev(B[0]), C, alpha=0.7, beta=-1.0, splits=splits, outer=(_dev(U), _dev(V), 0.25))
    assert _nrel(C.cpu().numpy(), 0.7 * A[0] @ B[0] - C0[0] + 0.25 * U.T @ V) < 1e-12


@pytest.mark.parametrize('M', [1, 15, 63, 64, 65, 128, 129, 200, 256])
@pytest.mark.parametrize('D,sets', [(1, 1), (3, 2)])
def test_moments(M, D, sets):
    from geepee_amd import dops
    print('moments', M, D, sets, flush=True)
    rs = np.random.RandomState(M)
    S, t = rs.randn(sets * D, M, M), rs.randn(D, M)
    mu, P = dops.moments(_dev(S), _dev(t), 0.5, -2.0)
    scale = np.repeat([0.5, -2.0][:sets], D)
    want = scale[:, None] * np.einsum('bij,bj->bi', S, np.tile(t, (sets, 1)))
    assert _nrel(mu.cpu().numpy(), want) < 1e-12
    assert _nrel(P.cpu().numpy(), S + want[:, :, None] * want[:, None, :]) < 1e-12


@pytest.mark.parametrize('M,Q', [(1, 1), (64, 5), (65, 16), (256, 8)])
def test_kuu_tail(M, Q):
    from geepee_amd import dops
    print('kuu tail', M, Q, flush=True)
    rs = np.random.RandomState(M + Q)
    Mm, z, ls, sf = [_dev(a) for a in (rs.randn(M, M), rs.randn(M, Q), 0.1 * rs.randn(Q) + 1.0, rs.randn(1) * 0.1)]
    dell, dsf2, sumdv, dz = [_dev(a) for a in (rs.randn(Q), rs.randn(1), rs.randn(1), rs.randn(M, Q))]
    gsf, gls, gz = dops.dtrace(Mm, z, ls, sf)
    want = dops.hyper(ls, sf, dell, gls, dsf2, sumdv, gsf) + (dz + gz,)
    got = dops.kuu_tail(Mm, z, ls, sf, dell, dsf2, sumdv, dz)
    for a, b in zip(got, want):
        assert _nrel(a.cpu().numpy(), b.cpu().numpy()) < 1e-12


@pytest.mark.parametrize('M,D', [(1, 1), (32, 3), (33, 17), (256, 2)])
def test_vfe_kl(M, D):
    from geepee_amd import _lib as L
    print('kl', M, D, flush=True)
    rs = np.random.RandomState(M)
    ldK, ldS, Ki, S = rs.randn(1), rs.randn(D), rs.randn(M, M), rs.randn(D, M, M)
    out, work = _dev(np.zeros(2)), _dev(np.zeros(L.query('gpx_vfe_kl_workspace', D, M)))
    d = [_dev(a) for a in (ldK, ldS, Ki, S)]
    L.call('gpx_vfe_kl_ws', D, M, L.P(d[0]), L.P(d[1]), -1.0, L.P(d[2]), L.P(d[3]), L.P(out), L.P(work), L.S())
    L.call('gpx_vfe_kl', D, M, L.P(d[0]), L.P(d[1]), -1.0, L.P(d[2]), L.P(d[3]), L.P(out[1:]), L.S())
    want = 0.5 * (D * ldK[0] + ldS.sum() - D * M + (Ki * S.sum(0)).sum())
    bar = 1e-12 * (abs(D * ldK[0]) + np.abs(ldS).sum() + D * M + np.abs(Ki * S.sum(0)).sum())
    assert np.all(np.abs(out.cpu().numpy() - want) < bar)
