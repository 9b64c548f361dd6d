"""The packed gradient w.r.t. theta1's factor at the edges of its tiles (GPU only).

Tolerance: sums of at most 256 products of order one: 1e-12 normwise.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('M', [1, 7, 8, 15, 16, 17, 31, 33, 50, 128, 129, 250, 256])
@pytest.mark.parametrize('D', [1, 3])
def test_pack_dR(M, D):
    from geepee_amd import dops
    print('pack', M, D, flush=True)
    rs = np.random.RandomState(M + D)
    R, G = np.triu(rs.randn(D, M, M)), rs.randn(D, M, M)
    P = R @ (G + G.transpose(0, 2, 1))
    P *= np.where(np.eye(M), R, 1.0)
    want = np.stack([p[np.triu_indices(M)] for p in P])
    got = dops.pack_dR(torch.as_tensor(R, device='cuda'), torch.as_tensor(G, device='cuda')).cpu().numpy()
    assert np.linalg.norm(got - want) < 1e-12 * np.linalg.norm(want)
