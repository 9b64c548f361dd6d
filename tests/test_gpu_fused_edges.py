"""The fused moment-matched kernels at the edges of their dispatch (GPU only): every count of
exponent slices (Q = 1 .. 16) and of output slices (D = 1 .. 32), partial 16-row tiles and
point blocks, the point counts per workgroup that fall back for lack of LDS, and far-away
points whose psi2 underflows.

Oracle: the moment-matching formulas in float64 on the CPU with torch's autograd.
Tolerance: an exponent of magnitude E carries an absolute error of a few E eps, E < 300 here, so
every psi2 entry is within 4 * 300 * 2.2e-16 = 2.7e-13 relative; sums of products of mixed
sign lose at most one to two digits more at these sizes: 1e-11 normwise.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _problem(N, M, Q, D, far=False):
    rs = np.random.RandomState(N + 7 * M + 11 * Q + 13 * D)
    t = lambda a: torch.as_tensor(a, dtype=torch.float64)
    mx, vx = t(rs.randn(N, Q)), t(rs.uniform(0.0, 0.5, (N, Q)))
    if far:
        mx[: (N + 1) // 2] += 60.0
    z, ls, sf = t(rs.randn(M, Q)), t(0.2 * rs.randn(Q) + 0.4), t(np.array([0.3]))
    B = rs.randn(D, M, M) / M
    return mx, vx, z, ls, sf, t(rs.randn(D, M)), t(0.5 * (B + B.transpose(0, 2, 1)))


def _reference(mx, vx, z, ls, sf, A, B):
    l = torch.exp(2 * ls)
    e1, e2 = 0.0, 0.0
    for q in range(mx.shape[1]):
        s1, s2 = l[q] + vx[:, q:q + 1], l[q] + 2 * vx[:, q, None, None]
        h = 0.5 * (z[:, None, q] + z[None, :, q])
        e1 = e1 + 0.5 * torch.log(l[q] / s1) - 0.5 * (mx[:, q:q + 1] - z[None, :, q]) ** 2 / s1
        e2 = e2 + 0.5 * torch.log(l[q] / s2) - (mx[:, q, None, None] - h) ** 2 / s2 \
            - (z[:, None, q] - z[None, :, q]) ** 2 / (4 * l[q])
    psi1, psi2 = torch.exp(2 * sf + e1), torch.exp(4 * sf + e2)
    m = psi1 @ A.T
    v = torch.exp(2 * sf) + torch.einsum('nab,dab->nd', psi2, B) - m ** 2
    return m, v


def _close(x, y):
    x, y = x.cpu(), y.detach()
    assert torch.isfinite(x).all()
    assert torch.linalg.norm(x - y) <= TOL * max(float(torch.linalg.norm(y)), 1e-300), \
        float(torch.linalg.norm(x - y) / torch.linalg.norm(y))


SHAPES = [(1, 1, 1, 1), (16, 16, 4, 4), (17, 15, 5, 5), (33, 17, 8, 8), (65, 40, 9, 9), (31, 33, 12, 16),
          (50, 31, 13, 17), (20, 48, 15, 32), (70, 130, 3, 2), (40, 250, 2, 3), (23, 256, 15, 4), (300, 20, 6, 31)]


@pytest.mark.parametrize('far', [False, True])
@pytest.mark.parametrize('N,M,Q,D', SHAPES)
def test_fused_edges(N, M, Q, D, far):
    from geepee_amd import dops
    print('fused edges', N, M, Q, D, far, flush=True)
    P = _problem(N, M, Q, D, far)
    rs = np.random.RandomState(5)
    gm, gv = (torch.as_tensor(rs.randn(N, D)) for _ in range(2))
    ins = [p.clone().requires_grad_(True) for p in P]
    m, v = _reference(*ins)
    dmx, dvx, dz, _, _, _, dB = torch.autograd.grad([m, v], ins, [gm, gv])
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    Bp = dops.sym_pairmajor(B)
    nt = (M + 15) // 16 * ((M + 15) // 16 + 1) // 2
    for nsub, splits in ((1, 1), (2, min(nt, 3)), (4, min(nt, 8))):
        plan = {'nsub': nsub, 'splits_f': splits, 'splits_b': 1, 'nsplit': nsub}
        psi1, mo, vo = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, Bp, plan=plan)
        _close(mo, m)
        _close(vo, v)
        dm = gm.cuda() - 2 * gv.cuda() * mo
        out = dops.fused_mm_bwd(mx, vx, z, ls, sf, A, Bp, psi1, dm, gv.cuda(), plan=plan)
        for got, want in zip((out[0], out[3], out[4], out[5]), (dB, dz, dmx, dvx)):
            _close(got, want)


def test_fused_forward_sixteen_inputs():
    from geepee_amd import dops
    P = _problem(19, 37, 16, 3)
    m, v = _reference(*P)
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    _, mo, vo = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, dops.sym_pairmajor(B))
    _close(mo, m)
    _close(vo, v)


@pytest.mark.parametrize('N,M,Q,D', [(1, 5, 1, 1), (17, 16, 3, 2), (40, 50, 15, 32), (33, 256, 4, 1), (20, 20, 16, 2),
                                     (9, 12, 2, 33)])
def test_posterior_propagation_without_psi2(N, M, Q, D):
    """forward_prop_thru_post at Gaussian inputs folds psi2 into the contraction where the fused
    kernels take the shape (Q <= 15, D <= 32); with return_info it stores psi2, and at the last
    two shapes it always does."""
    from geepee_amd.layers import SGP_Layer
    P = _problem(N, M, Q, D)
    L = SGP_Layer(100, Q, D, M)
    mx, vx, L.zu, L.ls, L.sf, L.A, L.B_sto = [p.cuda().contiguous() for p in P]
    L._pred_ready, L._Bp_post = True, None
    m, v = L.forward_prop_thru_post(mx, vx)
    m2, v2, psi1, psi2 = L.forward_prop_thru_post(mx, vx, return_info=True)
    assert psi1.shape == (N, M) and psi2.shape == (N, M, M)
    for got in ((m, v), (m2, v2)):
        for x, y in zip(got, _reference(*P)):
            _close(x, y)


def _far_rows(mx, vx):
    """Rows whose psi2 is an exact 0: infinite and huge means and variances."""
    inf = float('inf')
    mx[0, 0], mx[1, -1], mx[2, 0], mx[3, -1] = inf, -inf, 1e40, -1e60
    vx[4, 0], vx[5, -1] = inf, 1e308
    mx[6, 0], vx[6, -1] = 1e35, inf if mx.shape[1] > 1 else 0.5


@pytest.mark.parametrize('Q,D', [(1, 1), (2, 3), (5, 6), (8, 17)])
@pytest.mark.parametrize('N,M', [(7, 3), (40, 33), (70, 130)])
def test_posterior_propagation_infinite_inputs(N, M, Q, D):
    """An infinite or huge mean or variance gives psi2 = 0, so mean 0 and variance sf2; the other
    rows are those of the call without it, and a NaN stays in its row."""
    from geepee_amd.layers import SGP_Layer
    print('far inputs', N, M, Q, D, flush=True)
    P = _problem(N, M, Q, D)
    L = SGP_Layer(100, Q, D, M)
    mx, vx, L.zu, L.ls, L.sf, L.A, L.B_sto = [p.cuda().contiguous() for p in P]
    L._pred_ready, L._Bp_post = True, None
    m0, v0 = L.forward_prop_thru_post(mx, vx)
    _far_rows(mx, vx)
    m, v = L.forward_prop_thru_post(mx, vx)
    assert m[:7].abs().max() < 1e-140, m[:7]
    torch.testing.assert_close(v[:7], torch.exp(2 * L.sf).expand(7, D), rtol=1e-15, atol=0.0)
    assert torch.equal(m[7:], m0[7:]) and torch.equal(v[7:], v0[7:])
    m2, v2, psi1, psi2 = L.forward_prop_thru_post(mx, vx, return_info=True)
    assert torch.equal(psi2[:7], torch.zeros_like(psi2[:7]))
    mx[0, 0], vx[1, 0] = float('nan'), float('nan')
    m, v = L.forward_prop_thru_post(mx, vx)
    assert torch.isnan(m[:2]).all() and torch.isnan(v[:2]).all()
    assert torch.isfinite(m[2:]).all() and torch.isfinite(v[2:]).all()


@pytest.mark.parametrize('N,M,Q,D', [(40, 33, 2, 3), (40, 20, 5, 6), (1003, 33, 3, 2)])
def test_fused_adjoint_huge_inputs(N, M, Q, D):
    """Points so far out that psi1 and psi2 are exact zeros contribute nothing to any gradient."""
    from geepee_amd import dops
    print('far adjoint', N, M, Q, D, flush=True)
    P = _problem(N, M, Q, D)
    rs = np.random.RandomState(6)
    dm, dv = (torch.as_tensor(rs.randn(N, D)).cuda() for _ in range(2))
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    Bp = dops.sym_pairmajor(B)
    mx[0, 0], mx[N - 1, -1] = 1e40, -1e50
    psi1, _, _ = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, Bp)
    got = dops.fused_mm_bwd(mx, vx, z, ls, sf, A, Bp, psi1, dm, dv)
    for x in got[4:]:
        assert torch.equal(x[0], torch.zeros_like(x[0])) and torch.equal(x[-1], torch.zeros_like(x[-1])), x[[0, -1]]
    cut = lambda x: x[1:-1].contiguous()
    want = dops.fused_mm_bwd(cut(mx), cut(vx), z, ls, sf, A, Bp, cut(psi1), cut(dm), cut(dv))
    for x, y in zip(got[:4], want[:4]):
        _close(x, y.cpu())


@pytest.mark.parametrize('N,M,Q,D', [(1, 250, 4, 2), (37, 256, 3, 5), (90, 200, 2, 17), (5, 70, 5, 1), (3000, 9, 2, 3),
                                     (2500, 16, 3, 20), (1500, 48, 2, 4)])
def test_fused_default_plan_extremes(N, M, Q, D):
    """The rule's own plan where it asks for the most splits (few points, many tiles) and the most
    point ranges (many points, few tiles)."""
    from geepee_amd import dops
    plan = dops.fused_plan(N, M, Q, D, tuned=False)
    print('default plan', N, M, Q, D, plan, flush=True)
    assert plan['splits_f'] > 8 or plan['nsplit'] >= 32
    P = _problem(N, M, Q, D)
    rs = np.random.RandomState(7)
    gm, gv = (torch.as_tensor(rs.randn(N, D)) for _ in range(2))
    ins = [p.clone().requires_grad_(True) for p in P]
    m, v = _reference(*ins)
    dmx, dvx, dz, _, _, _, dB = torch.autograd.grad([m, v], ins, [gm, gv])
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    Bp = dops.sym_pairmajor(B)
    psi1, mo, vo = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, Bp, plan=plan)
    _close(mo, m)
    _close(vo, v)
    out = dops.fused_mm_bwd(mx, vx, z, ls, sf, A, Bp, psi1, gm.cuda() - 2 * gv.cuda() * mo, gv.cuda(), plan=plan)
    for got, want in zip((out[0], out[3], out[4], out[5]), (dB, dz, dmx, dvx)):
        _close(got, want)


def test_lengthscale_gradient_error():
    """dell sums a thousand points' terms of both signs; its relative error against extended precision,
    root mean square over ten problems, stays within 2.2 eps (one running sum over the blocks and a
    reciprocal in place of each point's divisions came to 2.6)."""
    from geepee_amd import dops
    L = np.longdouble
    N, M, Q, D = 1030, 20, 3, 3
    errs = []
    for seed in range(10):
        rs = np.random.RandomState(1000 + seed)
        mx, vx, z = rs.randn(N, Q), rs.uniform(0.02, 0.5, (N, Q)), 1.2 * rs.randn(M, Q)
        ls, sf = 0.15 * rs.randn(Q) + 0.1 + 0.1 * np.sqrt(Q), np.array([0.2])
        B = rs.randn(D, M, M) / M
        A, dm, dv = rs.randn(D, M), rs.randn(N, D), rs.randn(N, D)
        B = 0.5 * (B + B.transpose(0, 2, 1))
        t = [torch.as_tensor(a, device='cuda') for a in (mx, vx, z, ls, sf, A)]
        Bp = dops.sym_pairmajor(torch.as_tensor(B, device='cuda'))
        psi1 = dops.fused_mm_fwd(*t, Bp)[0]
        got = dops.fused_mm_bwd(*t, Bp, psi1, torch.as_tensor(dm, device='cuda'), torch.as_tensor(dv, device='cuda'))[2]
        mx, vx, z, l = mx.astype(L), vx.astype(L), z.astype(L), np.exp(2 * ls.astype(L))
        sf2 = np.exp(2 * sf.astype(L))[0]
        e1, e2, g1, g2 = 0, 0, [], []
        for q in range(Q):
            s1, s2 = (l[q] + vx[:, q])[:, None], (l[q] + 2 * vx[:, q])[:, None, None]
            u = (mx[:, q, None] - z[None, :, q]) ** 2
            w = (mx[:, q, None, None] - (z[:, None, q] + z[None, :, q]) / 2) ** 2
            dd = (z[:, None, q] - z[None, :, q]) ** 2
            e1 = e1 + np.log(l[q] / s1) / 2 - u / s1 / 2
            e2 = e2 + np.log(l[q] / s2) / 2 - w / s2 - dd / (4 * l[q])
            g1.append(1 / (2 * l[q]) - 1 / s1 / 2 + u / s1 ** 2 / 2)
            g2.append(1 / (2 * l[q]) - 1 / s2 / 2 + dd / (4 * l[q] ** 2) + w / s2 ** 2)
        L1 = dm.astype(L) @ A.astype(L) * sf2 * np.exp(e1)
        L2 = (dv.astype(L) @ B.reshape(D, -1).astype(L)).reshape(N, M, M) * sf2 ** 2 * np.exp(e2)
        want = np.array([((L1 * a).sum() + (L2 * b).sum()) * 2 * np.exp(ls.astype(L)[q])
                         for q, (a, b) in enumerate(zip(g1, g2))])
        errs.append(float(np.sqrt(((got.cpu().numpy().astype(L) - want) ** 2).sum() / (want ** 2).sum())))
    rms = np.sqrt(np.mean(np.square(errs)))
    print('dell error', rms / 2.0 ** -52, 'eps', flush=True)
    assert rms < 2.2 * 2.0 ** -52
