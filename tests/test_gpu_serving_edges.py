"""The grouped predict kernel at the edges of its dispatch (GPU only): several outputs in either
layer, more outputs than one pass of the first layer takes, hidden widths on both sides of
four, partial 16-row tiles, M at its limits.  Oracle: the float64 predictive with the bar of
the other serving tests (1e-9, or ten times the oracle's own LU-against-Cholesky spread)."""
import numpy as np
import pytest

from oracle import aep_oracle as O
from geepee_amd import workloads as W

pytestmark = pytest.mark.gpu


def _nrel(a, b):
    return np.linalg.norm(np.ravel(a - b)) / max(np.linalg.norm(np.ravel(b)), 1e-300)


def _spec(rs, M, Din, H, Dout):
    x = rs.randn(4 * M + 8, Din)
    if H == 0:
        p = W.layer_params(rs, Din, Dout, M, x=x)
        sp = dict(kind='sgpr', Din=Din, Ms=[M], N=len(x), hidden=[], Dout=Dout, params=p)
    else:
        p = W.layer_params(rs, Din, H, M, x=x, sfx='_0')
        p.update(W.layer_params(rs, H, Dout, M, sfx='_1', ls=np.log(1.0), sf=np.log(1.0)))
        sp = dict(kind='sdgpr', Din=Din, Ms=[M, M], N=len(x), hidden=[H], Dout=Dout, params=p)
    p['sn'] = np.array([np.log(0.1)])
    return sp


def _oracle(sp, X):
    def one():
        if sp['kind'] == 'sgpr':
            return O.sgpr_predict(sp['params'], sp['Ms'][0], sp['N'], X, noisy=True)
        return O.sdgpr_predict(sp['params'], sp['Ms'], sp['N'], X, noisy=True)
    O.INV = 'lu'
    want = one()
    O.INV = 'chol'
    try:
        alt = one()
    finally:
        O.INV = 'lu'
    return [(w, max(1e-9, 10 * _nrel(a, w))) for w, a in zip(want, alt)]


# (M, Din, hidden width or 0, Dout)
MODELS = [(1, 2, 0, 1), (15, 16, 0, 3), (16, 5, 0, 8), (33, 6, 0, 11), (17, 9, 8, 3), (40, 7, 5, 16), (31, 8, 4, 1),
          (48, 6, 1, 2), (250, 10, 3, 1), (256, 12, 8, 2)]


def test_serving_edges():
    from geepee_amd.serving import ModelStore
    rs = np.random.RandomState(11)
    specs = [_spec(rs, *m) for m in MODELS]
    store = ModelStore(specs)
    reqs = [(i, rs.randn(n, specs[i]['Din'])) for i in range(len(specs)) for n in (1, 16, 21)]
    outs = store.predict_many(reqs, noisy=True)
    for (i, X), got in zip(reqs, outs):
        print('serving edge', MODELS[i], len(X), flush=True)
        for g, (w, bar) in zip(got, _oracle(specs[i], X)):
            assert g.shape == w.shape and _nrel(g, w) < bar, (MODELS[i], len(X), _nrel(g, w), bar)
    alone = store.predict_many([reqs[14]], noisy=True)[0]
    assert all(np.array_equal(a, b) for a, b in zip(alone, outs[14]))
