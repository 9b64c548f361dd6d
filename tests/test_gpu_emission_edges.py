"""The linear-Gaussian emission over its register forms and block edges (GPU only).

Tolerance: Vy is R/alpha (0.08 to 0.72) plus C diag(vx) C^T (at most about 16 here), condition
about 200, so with up to 8 outputs per-step results are good to about 200 * 8 * 4 ulp = 1.5e-12
of the largest; 1e-11 is taken, for the sums over the steps relative to the sum of magnitudes.
"""
import numpy as np
import pytest
import torch

from oracle import aep_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Nb', [1, 64, 65, 4161])
@pytest.mark.parametrize('Dout,Din', [(1, 1), (8, 4), (8, 5), (8, 8), (3, 7), (2, 9), (7, 9), (1, 64)])
def test_emission(Nb, Dout, Din):
    from geepee_amd import dops
    print('emission', Nb, Dout, Din, flush=True)
    rs = np.random.RandomState(Nb + 10 * Dout + Din)
    alpha, scale = 0.5, -3.0
    C, Rp = rs.randn(Dout, Din), np.log(rs.uniform(0.2, 0.6, Dout))
    y, mx, vx = rs.randn(Nb, Dout), rs.randn(Nb, Din), rs.uniform(0.1, 0.5, (Nb, Din))
    lz, gin, gh = O.emission_tilted(C, Rp, y, mx, vx, alpha, scale)
    # magnitudes of the terms of the sums
    R = np.exp(2 * Rp)
    Vy = np.diag(R / alpha) + np.einsum('ac,nc,bc->nab', C, vx, C)
    Vi = np.linalg.inv(Vy)
    r = y - mx @ C.T
    u = np.einsum('nab,nb->na', Vi, r)
    dS = -0.5 * Vi + 0.5 * u[:, :, None] * u[:, None, :]
    magC = (np.abs(u)[:, :, None] * np.abs(mx)[:, None, :] + 2 * np.abs(dS @ C) * vx[:, None, :]).sum(0).max()
    magR = ((0.5 * np.diagonal(Vi, axis1=1, axis2=2) + 0.5 * u ** 2).sum(0).max() / alpha + 0.5 * Nb / R.min()) * 2 * R.max()
    magZ = np.abs(r * u).sum() + np.abs(np.linalg.slogdet(Vy)[1]).sum() + Nb * Dout * (4 + np.abs(np.log(R)).max())
    t = [torch.as_tensor(a, device='cuda') for a in (C, Rp, y, mx, vx)]
    dmx, dvx, dC, dR, scal = [a.cpu().numpy() for a in dops.emission(*t, alpha, scale)]
    assert np.abs(dmx - gin['mx']).max() < 1e-11 * np.abs(gin['mx']).max()
    assert np.abs(dvx - gin['vx']).max() < 1e-11 * np.abs(gin['vx']).max()
    assert np.abs(dC - gh['C']).max() < 1e-11 * abs(scale) * magC
    assert np.abs(dR - gh['R']).max() < 1e-11 * abs(scale) * magR
    assert abs(scal[0] - lz) < 1e-11 * abs(scale) * magZ
