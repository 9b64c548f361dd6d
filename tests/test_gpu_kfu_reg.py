"""The kernel matrix's adjoint with its gradient formed on the fly (GPU only): against the separate
product, weighted sum and adjoint, over column layouts, register widths, outputs and odd row counts.

Tolerance: the same sums in another order, terms of mixed sign: 1e-11 normwise.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,D,M,Q', [(1, 1, 1, 1), (3, 2, 64, 4), (33, 3, 65, 5), (130, 1, 128, 8), (7, 5, 129, 9),
                                     (1000, 4, 100, 12), (257, 33, 40, 13), (2049, 2, 256, 16), (20001, 1, 50, 2)])
def test_kfu_reg(N, D, M, Q):
    from geepee_amd import dops
    print('kfu reg', N, D, M, Q, flush=True)
    rs = np.random.RandomState(N + D + M + Q)
    t = lambda *s: torch.as_tensor(rs.randn(*s), device='cuda')
    dm, dv, A, T, x, z = t(N, D), t(N, D), t(D, M), t(D, N, M), t(N, Q), t(M, Q)
    ls, sf = 0.2 * t(Q) + 0.5, 0.1 * t(1)
    K = dops.se(x, z, ls, sf)
    dK = dops.mm(dm, A)
    dops.wsum(dv, T, dK, alpha=2.0, beta=1.0)
    dsf2, dell, dz, _ = dops.kfu_bwd(dK, K, x, z, ls, sf)
    got = dops.kfu_bwd_reg(dm, dv, A, T, K, x, z, ls, sf)
    scale = float((dK * K).abs().sum() / torch.exp(2 * sf)) + float(dv.abs().sum())
    assert abs(float(got[0]) - float(dsf2) - float(dv.sum())) < 1e-11 * scale
    for a, b in ((got[1], dell), (got[2], dz)):
        assert float((a - b).norm()) <= 1e-11 * float(b.norm())
