"""The Gaussian tilted likelihood around its block counts and sizes (GPU only).

Tolerance: per-element formulas to a few ulp (1e-13), the two sums of up to 70000 terms of one sign
or mixed within 1e-12 of the sum of magnitudes.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,D', [(1, 1), (256, 1), (257, 1), (5462, 3), (16384, 1), (16385, 1), (17500, 4)])
@pytest.mark.parametrize('alpha', [1.0, 0.3])
def test_gauss_tilted(B, D, alpha):
    from geepee_amd import dops
    print('tilted', B, D, alpha, flush=True)
    rs = np.random.RandomState(B + D)
    m, v, y, sn, scale = rs.randn(B, D), rs.rand(B, D) + 0.1, rs.randn(B, D), np.array([-0.7]), 0.37
    sn2 = np.exp(2 * sn[0])
    vt, r = v + sn2 / alpha, y - m
    gm, gv = r / vt, -0.5 / vt + 0.5 * r * r / vt ** 2
    terms = -0.5 * (np.log(2 * np.pi * vt) + r * r / vt)
    const = B * D * (0.5 * np.log(2 * np.pi * sn2 / alpha) - 0.5 * alpha * np.log(2 * np.pi * sn2))
    t = [torch.as_tensor(a, device='cuda') for a in (m, v, y, sn)]
    dm, dv, dmall, scal = [a.cpu().numpy() for a in dops.gauss_tilted(*t, alpha, scale, want_dmall=True)]
    assert np.allclose(dm, scale * gm, rtol=1e-13, atol=1e-15)
    assert np.allclose(dv, scale * gv, rtol=1e-12, atol=1e-14)
    assert np.allclose(dmall, scale * gm - 2 * scale * gv * m, rtol=1e-11, atol=1e-13)
    assert abs(scal[0] - (terms.sum() + const)) < 1e-12 * (np.abs(terms).sum() + abs(const))
    dsn = (gv.sum() * 2 * sn2 / alpha + B * D * (1 - alpha)) * scale
    assert abs(scal[1] - dsn) < 1e-12 * (np.abs(gv).sum() * 2 * sn2 / alpha + B * D) * scale


def test_gauss_tilted_mean_gradient_is_one_division():
    """With unit noise and alpha = 1 the mean's gradient is (y - m) / (v + 1), correctly rounded."""
    from geepee_amd import dops
    rs = np.random.RandomState(3)
    m, v, y = rs.randn(3000, 3), rs.rand(3000, 3) + 0.01, rs.randn(3000, 3)
    t = [torch.as_tensor(a, device='cuda') for a in (m, v, y, np.zeros(1))]
    dm = dops.gauss_tilted(*t, 1.0, 1.0)[0].cpu().numpy()
    assert np.array_equal(dm, (y - m) / (v + 1.0))


@pytest.mark.parametrize('n', [16384, 16385, 20001, 65536, 65537, 75052, 131072, 131073])
def test_x_gradients_over_thread_counts(n):
    """Each latent element's gradient is the same bits whatever the launch shape (a slice of the rows
    gives the slice's), and the sum of log-normalisers is that of the slices; the same for the
    transition terms."""
    from geepee_amd import dops, xfactors as X
    print('x gradients', n, flush=True)
    rs = np.random.RandomState(n)
    dev = lambda *s: torch.as_tensor(rs.randn(*s), device='cuda')
    x1, x2, gm, gv = dev(n, 1), 0.3 * dev(n, 1), dev(n, 1), dev(n, 1)
    args = (0.6, 0.2, 1.5)

    def lvm(a, b):
        xs = X.lvm_x_state(x1[a:b].contiguous(), x2[a:b].contiguous(), None, *args, False)
        g1, g2, s = X.lvm_x_grads(xs, gm[a:b], gv[a:b], b - a, b - a, *args, 1, False)
        return g1, g2, float(s[0])

    cuts = list(range(0, n, 9001)) + [n]
    whole, parts = lvm(0, n), [lvm(a, b) for a, b in zip(cuts, cuts[1:])]
    for k in (0, 1):
        assert torch.equal(whole[k], torch.cat([p[k] for p in parts]))
    assert abs(whole[2] - sum(p[2] for p in parts)) < 1e-12 * n
    t = [dev(n, 1), dev(n, 1).abs() + 0.1, dev(n, 1), dev(n, 1).abs() + 0.1]
    sn = torch.zeros(1, dtype=torch.float64, device='cuda')
    full = dops.transition(*t, sn, 0.6, 1.0)
    part = [dops.transition(*[u[a:b].contiguous() for u in t], sn, 0.6, 1.0) for a, b in zip(cuts, cuts[1:])]
    for k in range(4):
        assert torch.equal(full[k], torch.cat([p[k] for p in part]))
    assert abs(float(full[4][0]) - sum(float(p[4][0]) for p in part)) < 1e-12 * n
