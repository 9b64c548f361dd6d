"""The adjoint of the psi statistics at the edges of its layout (GPU only): 16-column tiles over
four or eight waves (M = 1 ... 256), groups of eight rows and their remainders, Q up to 16, fewer
and more points than workgroups, symmetric and general dL/dpsi2.

Reference: torch autograd (float64, CPU) of the closed forms.  Tolerance: every output is a sum of
at most N M^2 < 2e5 rounded terms, with differences (m S0 - S1 and the like) that lose up to three
digits: 2e5^(1/2) * 1.1e-16 * 1e3 < 1e-10 normwise.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _psi(mx, vx, z, ls, sf):
    l = torch.exp(2 * ls)
    sf2 = torch.exp(2 * sf)
    d1 = mx[:, None] - z[None]
    psi1 = sf2 * torch.exp((0.5 * torch.log(l / (l + vx))).sum(1)[:, None] - (d1 ** 2 / (2 * (l + vx))[:, None]).sum(2))
    dz = z[:, None] - z[None]
    mid = 0.5 * (z[:, None] + z[None])
    lead = (0.5 * torch.log(l / (l + 2 * vx))).sum(1)[:, None, None] - (dz ** 2 / (4 * l)).sum(2)[None]
    far = ((mx[:, None, None] - mid[None]) ** 2 / (2 * vx + l)[:, None, None]).sum(3)
    return psi1, sf2 ** 2 * torch.exp(lead - far)


def _nrel(a, b):
    return float((a.cpu() - b).norm() / b.norm().clamp_min(1e-300))


@pytest.mark.parametrize('N,M,Q', [(1, 1, 1), (3, 7, 2), (5, 8, 4), (4, 16, 5), (800, 15, 3), (9, 33, 16), (6, 64, 8),
                                   (3, 65, 9), (3, 100, 12), (2, 128, 1), (2, 129, 13), (1, 200, 16), (2, 256, 4)])
def test_psi_adjoint(N, M, Q):
    from geepee_amd import dops
    from geepee_amd.autograd import psi_statistics
    print('psi adjoint', N, M, Q, flush=True)
    g = torch.Generator().manual_seed(N + M + Q)
    rn = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)
    par = [rn(N, Q), torch.rand(N, Q, generator=g, dtype=torch.float64) + 0.1, rn(M, Q), 0.2 * rn(Q) + 0.5 * Q ** 0.5,
           0.2 * rn(1)]
    g1, g2 = rn(N, M), rn(N, M, M)
    ref = [p.clone().requires_grad_() for p in par]
    p1, p2 = _psi(*ref)
    want = torch.autograd.grad((p1 * g1).sum() + (p2 * g2).sum(), ref)
    dev = [p.cuda().requires_grad_() for p in par]
    d1, d2 = psi_statistics(*dev)
    got = torch.autograd.grad((d1 * g1.cuda()).sum() + (d2 * g2.cuda()).sum(), dev)
    for a, b in zip(got, want):
        assert _nrel(a, b) < 1e-10
    # a symmetric dL/dpsi2 through the entry point that reads it once
    gs = (0.5 * (g2 + g2.transpose(1, 2))).contiguous().cuda()
    dsf2, dell, dz, dmx, dvx = dops.psi_bwd(*[p.cuda() for p in par], g1.cuda(), d1.detach(), gs, d2.detach())
    for a, b in ((dmx, want[0]), (dvx, want[1]), (dz, want[2]), (dell.cpu() * torch.exp(par[3]), want[3]),
                 (dsf2.cpu() * 2 * torch.exp(2 * par[4]), want[4])):
        assert _nrel(a, b) < 1e-10
