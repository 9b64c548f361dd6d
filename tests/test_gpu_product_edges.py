"""Matrix products and weighted Gram matrices at the edges of their tiles (GPU only): 16-row and
16-column tiles, column bands of 1 to 4 tiles, k groups of 8 and their remainders, one or four
waves per tile, split K.

Tolerance: a sum of k <= 2000 products in any order is within k eps (< 5e-13) of the exact one
relative to the sum of magnitudes; the entries compared normwise are sums of random signs, which
loses at most sqrt(k) < 50 of that bound and in practice gains it back: 1e-12.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _nrel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize('tile', [0, 32, 64])
@pytest.mark.parametrize('m,n,k,b', [(1, 2, 2, 1), (15, 17, 7, 3), (16, 16, 8, 1), (33, 31, 9, 2), (64, 65, 40, 9),
                                     (100, 13, 257, 1), (7, 200, 2000, 4), (129, 80, 33, 5), (2100, 208, 72, 4)])
def test_gemm_edges(m, n, k, b, tile):
    from geepee_amd import _lib as L
    rs = np.random.RandomState(m + n + k + b)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device='cuda')
    for tA in (0, 1):
        for tB in (0, 1):
            A, B = rs.randn(b, *((k, m) if tA else (m, k))), rs.randn(*((n, k) if tB else (k, n)))
            C0, E = rs.randn(b, m, n), rs.randn(m, n)
            P = np.matmul(A.swapaxes(1, 2) if tA else A, B.T if tB else B)
            for splits in (1, 3):
                print('gemm', m, n, k, b, tile, tA, tB, splits, flush=True)
                C = dev(C0)
                L.mm(dev(A), dev(B), C, tA=bool(tA), tB=bool(tB), alpha=0.7, beta=-0.5, splits=splits, tile=tile,
                     E=dev(E), gamma=2.0)
                assert _nrel(C.cpu().numpy(), 0.7 * P - 0.5 * C0 + 2.0 * E) < 1e-12


@pytest.mark.parametrize('N,D,M', [(1, 1, 1), (7, 3, 15), (8, 1, 16), (9, 2, 17), (33, 5, 64), (63, 1, 65), (64, 2, 80),
                                   (65, 1, 81), (300, 3, 100), (500, 2, 144), (1999, 1, 200), (700, 2, 256)])
def test_gram_edges(N, D, M):
    from geepee_amd import dops
    rs = np.random.RandomState(N + D + M)
    w, X, E = rs.randn(N, D), rs.randn(N, M), rs.randn(D, M, M)
    ref = np.einsum('nd,na,nb->dab', w, X, X)
    dw, dX, dE = [torch.as_tensor(a, device='cuda') for a in (w, X, E)]
    for splits in (None, 1, 3, 16):
        print('gram', N, D, M, splits, flush=True)
        got = dops.gram(dw, dX, splits=splits).cpu().numpy()
        assert _nrel(got, ref) < 1e-12
        assert np.array_equal(got, got.swapaxes(1, 2))
    assert _nrel(dops.gram(dw, dX, E=dE, gamma=-0.5).cpu().numpy(), ref - 0.5 * E) < 1e-12
    assert _nrel(dops.gram(dw, dX, E=dE[0].contiguous(), gamma=1.0).cpu().numpy(), ref + E[:1]) < 1e-12
    assert not dops.gram(dw[:0], dX[:0]).any()


# (tiles of 32 x 32, k) on both sides of each line of the rule that gives a tile to a wave or to four
@pytest.mark.parametrize('k', [16, 17, 64, 65, 256, 257])
@pytest.mark.parametrize('tiles', [576, 577, 768, 769, 896, 897, 1024, 1025, 1536, 1537, 1792, 1793, 4095, 4096])
def test_gemm_wave_rule(tiles, k):
    from geepee_amd import _lib as L
    rs = np.random.RandomState(tiles + k)
    print('gemm rule', tiles, k, flush=True)
    A, B = rs.randn(32 * tiles - 5, k), rs.randn(k, 27)
    C = torch.full((A.shape[0], 27), float('nan'), dtype=torch.float64, device='cuda')
    L.mm(torch.as_tensor(A, device='cuda'), torch.as_tensor(B, device='cuda'), C, tile=32)
    assert _nrel(C.cpu().numpy(), A @ B) < 1e-12
