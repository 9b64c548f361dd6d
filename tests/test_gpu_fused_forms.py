"""Every form of the fused adjoint's contractions (GPU only): 4 x 4 products of one to three
groups against 16 x 16 tiles, on both sides of each line of the dispatch (Q = 3 | 4 | 7 | 8 | 11 | 12,
D = 4 | 8 | 12 | 16), a tile with rows past M and one without, a partial last point block.

Oracle and tolerance as for the other edges of these kernels: float64 autograd on the CPU, 1e-11
normwise.
"""
import numpy as np
import pytest
import torch

from tests.test_gpu_fused_edges import _close, _problem, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Q', [3, 4, 7, 8, 11, 12])
@pytest.mark.parametrize('D', [4, 5, 8, 9, 12, 13, 17])
def test_adjoint_forms(Q, D):
    from geepee_amd import dops
    N, M = 19, 32 if (Q + D) % 2 else 27
    print('fused forms', N, M, Q, D, flush=True)
    P = _problem(N, M, Q, D)
    rs = np.random.RandomState(Q + D)
    gm, gv = (torch.as_tensor(rs.randn(N, D)) for _ in range(2))
    ins = [p.clone().requires_grad_(True) for p in P]
    m, v = _reference(*ins)
    want = torch.autograd.grad((m * gm).sum() + (v * gv).sum(), ins)
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    Bp = dops.sym_pairmajor(B)
    psi1, mo, vo = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, Bp)
    _close(mo, m)
    _close(vo, v)
    dv = gv.cuda()
    dm_all = dops.dmall(gm.cuda(), dv, mo)
    dB, dsf2, dell, dz, dmx, dvx = dops.fused_mm_bwd(mx, vx, z, ls, sf, A, Bp, psi1, dm_all, dv)
    for got, ref in ((dmx, want[0]), (dvx, want[1]), (dz, want[2]), (dell.cpu() * torch.exp(P[3]), want[3]),
                     (0.5 * (dB + dB.transpose(1, 2)), 0.5 * (want[6] + want[6].transpose(1, 2)))):
        _close(got, ref)
    sf2 = torch.exp(2 * P[4])
    _close((dsf2.cpu() + gv.sum()) * 2 * sf2, want[4])


@pytest.mark.parametrize('nsplit', [2, 4])
@pytest.mark.parametrize('M', [64, 65, 128, 129, 192, 193])
@pytest.mark.parametrize('Q', [1, 4, 5, 8, 9, 12, 13, 15])
def test_row_finish_forms(Q, M, nsplit):
    """Every form of the row finish (slices of four inputs, column tiles a wave; at Q = 15 a 17th
    partial column), with a last point range of one point (2) and an empty one (4)."""
    from geepee_amd import dops
    N, D = 33, 3
    print('row finish', Q, M, nsplit, flush=True)
    P = _problem(N, M, Q, D)
    rs = np.random.RandomState(Q + M)
    gm, gv = (torch.as_tensor(rs.randn(N, D)) for _ in range(2))
    ins = [p.clone().requires_grad_(True) for p in P]
    m, v = _reference(*ins)
    want = torch.autograd.grad((m * gm).sum() + (v * gv).sum(), ins)
    mx, vx, z, ls, sf, A, B = [p.cuda() for p in P]
    Bp = dops.sym_pairmajor(B)
    plan = dict(dops.fused_plan(N, M, Q, D, tuned=False), nsplit=nsplit)
    psi1, mo, _ = dops.fused_mm_fwd(mx, vx, z, ls, sf, A, Bp, plan=plan)
    dm_all = dops.dmall(gm.cuda(), gv.cuda(), mo)
    dB, dsf2, dell, dz, dmx, dvx = dops.fused_mm_bwd(mx, vx, z, ls, sf, A, Bp, psi1, dm_all, gv.cuda(), plan=plan)
    for got, ref in ((dmx, want[0]), (dvx, want[1]), (dz, want[2]), (dell.cpu() * torch.exp(P[3]), want[3]),
                     (dB, want[6]), ((dsf2.cpu() + gv.sum()) * 2 * torch.exp(2 * P[4]), want[4])):
        _close(got, ref)
