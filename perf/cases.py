"""Timed workloads of the sparse-GP approximate-EP framework, through its public entry points.

Each case is one call that a user's program makes over and over: an energy+gradient
evaluation of a model (eagerly or replayed as a hipGraph, as the device-resident optimiser
does), a moment-matched layer or the psi statistics as differentiable functions, a
prediction, a batch of served requests.  Everything is IEEE double precision.

  listed()            the fixed cases
  draw(rng)           another case of the same ranges
  prepare(case, seed) inputs, parameters and handles, made from the seed alone
  run(state)          one pass, with all of its outputs
  work(case)          bytes and floating-point operations a pass cannot do without
  exact(case, seed)   the same outputs from plain torch in float64
"""
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

JITTER = 1e-5          # added to Kuu's diagonal by the framework
F64 = torch.float64


def listed():
    return [
        # the smallest training step: a low-dimensional regression with few inducing points,
        # replayed as a hipGraph (what optimise_device does per iteration)
        dict(name='sgpr_small', kind='sgpr', N=1000, M=50, Din=2, Dout=1, vfe=False, graph=True),
        # regression over a large full batch: the deterministic-input layer's long contractions
        dict(name='sgpr_large', kind='sgpr', N=20000, M=200, Din=8, Dout=4, vfe=False, graph=False),
        # the variational bound with as many inducing points as the layers take
        dict(name='vfe_sgpr', kind='sgpr', N=4001, M=256, Din=10, Dout=2, vfe=True, graph=True),
        # latent-variable model of the benchmark: psi2 recomputed in the fused kernels
        dict(name='sgplvm_fused', kind='sgplvm', N=4096, M=128, Q=8, D=32, fused=True, graph=True),
        # the same model as it comes without set_fused(): psi2 stored; ordinary data-set size
        dict(name='sgplvm_plain', kind='sgplvm', N=1000, M=100, Q=5, D=12, fused=False, graph=False),
        # three-layer deep GP on a batch of 1000 rows, replayed as a hipGraph
        dict(name='sdgpr_deep', kind='sdgpr', N=1000, M=100, Din=10, H=5, L=3, graph=True),
        # state-space model over a long series, replayed as a hipGraph
        dict(name='sgpssm_long', kind='sgpssm', T=10000, M=200, Din=4, Dout=8, graph=True),
        # a small moment-matched layer, forward only (scoring a handful of uncertain inputs)
        dict(name='mm_forward', kind='mm', N=301, M=40, Q=3, D=3, grad=False),
        # a wide moment-matched layer as a differentiable function, ragged sizes
        dict(name='mm_train', kind='mm', N=3001, M=190, Q=10, D=12, grad=True),
        # the psi statistics themselves as a differentiable function (psi2 is an output)
        dict(name='psi_train', kind='psi', N=1501, M=100, Q=5),
        # prediction of a fitted two-layer deep GP at a few thousand host-side inputs
        dict(name='predict_deep', kind='predict', N=5000, M=100, Din=8, H=4),
        # one admission of the prediction server: requests of mixed size over resident models
        dict(name='serve_mixed', kind='serve', models=32, requests=24, most=4096),
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(['sgpr', 'sgpr', 'sgplvm', 'sgplvm', 'sdgpr', 'sgpssm', 'mm', 'mm', 'mm', 'psi',
                           'predict', 'serve'])
        if kind == 'sgpr':
            c = dict(kind=kind, N=_between(rng, 200, 20000), M=_between(rng, 16, 256), Din=rng.randint(3, 10),
                     Dout=rng.randint(1, 4), vfe=rng.random() < 0.5, graph=rng.random() < 0.5)
        elif kind == 'sgplvm':
            fused = rng.random() < 0.6
            c = dict(kind=kind, N=_between(rng, 150, 4500 if fused else 1500), M=_between(rng, 20, 160),
                     Q=rng.randint(3, 10), D=_between(rng, 2, 32), fused=fused, graph=fused)
        elif kind == 'sdgpr':
            c = dict(kind=kind, N=_between(rng, 200, 3000), M=_between(rng, 20, 130), Din=rng.randint(4, 10),
                     H=rng.randint(3, 6), L=rng.randint(2, 3), graph=True)
        elif kind == 'sgpssm':
            c = dict(kind=kind, T=_between(rng, 300, 10000), M=_between(rng, 20, 200), Din=rng.randint(3, 5),
                     Dout=rng.randint(2, 8), graph=True)
        elif kind == 'mm':
            c = dict(kind=kind, N=_between(rng, 50, 8000), M=_between(rng, 16, 256), Q=rng.randint(2, 12),
                     D=_between(rng, 1, 32), grad=rng.random() < 0.7)
        elif kind == 'psi':
            c = dict(kind=kind, N=_between(rng, 100, 2000), M=_between(rng, 16, 160), Q=rng.randint(1, 10))
        elif kind == 'predict':
            c = dict(kind=kind, N=_between(rng, 1, 8000), M=_between(rng, 20, 160), Din=rng.randint(3, 10),
                     H=rng.randint(3, 5))
        else:
            c = dict(kind=kind, models=rng.randint(8, 48), requests=rng.randint(1, 30),
                     most=_between(rng, 4, 4096))
        # inducing points are a summary of the data: at most a quarter of its rows
        rows = c.get('T', c.get('N'))
        if kind in ('sgpr', 'sgplvm', 'sdgpr', 'sgpssm') and 4 * c['M'] > rows:
            c['M'] = max(16, rows // 4)
        if _cost(c) <= limit:
            return c


# ---------------------------------------------------------------------------
# inputs (numpy, from the seed alone)
# ---------------------------------------------------------------------------

def _spread(rs, x, M):
    """M inducing inputs: a farthest-point subset of the rows of x (spread over the data as
    k-means centres are), jittered."""
    if x.shape[0] < M:
        x = np.vstack([x, rs.randn(M - x.shape[0], x.shape[1])])
    c = x[rs.permutation(x.shape[0])[:4 * M]]
    d = np.full(c.shape[0], np.inf)
    pick = [0]
    for _ in range(M - 1):
        d = np.minimum(d, ((c - c[pick[-1]]) ** 2).sum(1))
        pick.append(int(d.argmax()))
    return c[pick] + 0.01 * rs.randn(M, x.shape[1])


def _layer(rs, Din, Dout, M, x, sfx='', sf=0.5):
    """Parameters of one layer: lengthscales about half the data's median distance (shorter
    where many inducing inputs share few dimensions), a full q(u) covariance."""
    med = math.sqrt(2.0 * x.var(0).sum())
    ell = 0.5 * med * min(1.0, 3.0 * M ** (-1.0 / Din))
    p = {'zu' + sfx: _spread(rs, x, M),
         'ls' + sfx: np.log(ell) + 0.1 * rs.randn(Din),
         'sf' + sfx: np.array([np.log(sf)])}
    iu = np.triu_indices(M)
    eta = 0.05 * rs.randn(Dout, iu[0].size)
    diag = iu[0] == iu[1]
    eta[:, diag] = np.log(1.0 / np.sqrt(0.5 * rs.rand(Dout, M) + 0.05))
    p['eta1_R' + sfx] = eta
    p['eta2' + sfx] = rs.randn(Dout, M)
    return p


def _inputs(case, seed):
    """(data arrays, parameter dict) of a case."""
    rs = np.random.RandomState(int(seed) % (1 << 32))
    k = case['kind']
    if k == 'sgpr':
        N, Din, Dout = case['N'], case['Din'], case['Dout']
        x = rs.uniform(-3, 3, (N, Din))
        y = np.sin(x).dot(rs.randn(Din, Dout)) + 0.1 * rs.randn(N, Dout)
        p = _layer(rs, Din, Dout, case['M'], x)
        p['sn'] = np.array([np.log(0.1)])
        return dict(x=x, y=y), p
    if k == 'sgplvm':
        N, Q = case['N'], case['Q']
        m, v = rs.randn(N, Q), rs.uniform(0.01, 0.5, (N, Q))
        y = np.tanh(m).dot(rs.randn(Q, case['D'])) + 0.3 * rs.randn(N, case['D'])
        p = _layer(rs, Q, case['D'], case['M'], m)
        p['sn'] = np.array([np.log(0.5)])
        p['x1'] = m / v
        p['x2'] = 0.5 * np.log(1.0 / v - 1.0)
        return dict(y=y), p
    if k in ('sdgpr', 'predict'):
        N, Din = case['N'], case['Din']
        L = case.get('L', 2)
        Ntr = N if k == 'sdgpr' else 4 * case['M']
        x = rs.randn(Ntr, Din)
        y = np.sin(x).sum(1, keepdims=True) + 0.05 * rs.randn(Ntr, 1)
        sizes = [Din] + [case['H']] * (L - 1) + [1]
        p = {}
        for i in range(L):
            xi = x if i == 0 else rs.randn(4 * case['M'], sizes[i])
            p.update(_layer(rs, sizes[i], sizes[i + 1], case['M'], xi, '_%d' % i, 0.5 if i == 0 else 1.0))
        p['sn'] = np.array([np.log(0.05)])
        return dict(x=x, y=y, sizes=sizes, xs=rs.randn(N, Din) if k == 'predict' else None), p
    if k == 'sgpssm':
        T, Din, Dout = case['T'], case['Din'], case['Dout']
        W = np.linalg.qr(rs.randn(Din, Din))[0]
        e = 0.3 * rs.randn(T, Din)
        xs = np.empty((T, Din))
        cur = rs.randn(Din)
        for t in range(T):
            cur = 0.9 * np.tanh(W.dot(cur)) + e[t]
            xs[t] = cur
        C = 0.5 * rs.randn(Dout, Din)
        y = xs.dot(C.T) + 0.1 * rs.randn(T, Dout)
        p = _layer(rs, Din, Din, case['M'], xs[:-1], '_dynamic')
        p['x_factor_1'] = xs / 0.1 / 3.0
        p['x_factor_2'] = 0.5 * math.log(1.0 / 0.1 / 3.0) + 0.1 * rs.randn(T, Din)
        p['C_emission'] = C + 0.05 * rs.randn(Dout, Din)
        p['R_emission'] = np.log(0.1) + 0.1 * rs.randn(Dout)
        p['sn'] = np.array([np.log(0.3)])
        return dict(y=y), p
    if k in ('mm', 'psi'):
        N, M, Q = case['N'], case['M'], case['Q']
        m = rs.randn(N, Q)
        d = dict(mx=m, vx=rs.uniform(0.01, 0.5, (N, Q)))
        p = _layer(rs, Q, 1, M, m)
        d.update(z=p['zu'], ls=p['ls'], sf=p['sf'])
        if k == 'mm':
            D = case['D']
            B = rs.randn(D, M, M) / M
            d.update(A=rs.randn(D, M) / math.sqrt(M), B=0.5 * (B + B.transpose(0, 2, 1)), gm=rs.randn(N, D),
                     gv=rs.randn(N, D))
        else:
            # dL/dpsi2 of a downstream layer: sum_d g_nd B_d
            g, B = rs.randn(N, 2), rs.randn(2, M, M) / M
            d.update(g1=rs.randn(N, M) / M, g2=g, B2=B)
        return d, None
    # serve: resident models of several sizes, requests of mixed length
    models, Ms = [], (32, 64, 128, 256)
    for i in range(case['models']):
        M, Din = Ms[i % 4], 3 + (7 * i) % 8
        x = rs.randn(4 * M, Din)
        if i % 2 == 0:
            p = _layer(rs, Din, 1, M, x)
            spec = dict(kind='sgpr', Din=Din, Ms=[M], N=4 * M, hidden=[], params=p)
        else:
            H = min(Din, 5)
            p = _layer(rs, Din, H, M, x, '_0')
            p.update(_layer(rs, H, 1, M, rs.randn(4 * M, H), '_1', 1.0))
            spec = dict(kind='sdgpr', Din=Din, Ms=[M, M], N=4 * M, hidden=[H], params=p)
        p['sn'] = np.array([np.log(0.1)])
        models.append(spec)
    reqs = [(i, rs.randn(n, models[i]['Din'])) for i, n in _requests(case)]
    return dict(models=models, reqs=reqs), None


def _requests(case):
    """(model, points) of each request: lengths log-uniform in [1, most], part of the case."""
    return [((7 * j + 3) % case['models'], max(1, int(math.exp((0.5 + 0.618 * j) % 1.0 * math.log(case['most'])))))
            for j in range(case['requests'])]


def _serve_work(case):
    """Floating-point operations and doubles in and out over the requests."""
    f = b = 0.0
    for i, n in _requests(case):
        M, Din = (32, 64, 128, 256)[i % 4], 3 + (7 * i) % 8
        H = min(Din, 5)
        f += n * (_det_flops(1, M, Din, 1, False) if i % 2 == 0
                  else _det_flops(1, M, Din, H, False) + _mm_flops(1, M, H, 1, False))
        b += n * (Din + 2)
    return f, b


ALPHA = 0.5


def prepare(case, seed):
    from geepee_amd import aep_models, vfe_models, graphs, serving
    d, p = _inputs(case, seed)
    k = case['kind']
    if k in ('mm', 'psi'):
        t = {n: torch.as_tensor(v, device='cuda') for n, v in d.items()}
        st = dict(kind=k, g=[])
        names = ['mx', 'vx', 'z', 'ls', 'sf'] + (['A', 'B'] if k == 'mm' else [])
        grad = k == 'psi' or case['grad']
        st['in'] = [t[n].requires_grad_(grad) for n in names]
        st['grad'] = grad
        if k == 'mm':
            st['up'] = [t['gm'], t['gv']]
        else:
            st['up'] = [t['g1'], torch.einsum('nd,dab->nab', t['g2'], t['B2']).contiguous()]
        return st
    if k == 'serve':
        return dict(kind=k, store=serving.ModelStore(d['models']), reqs=d['reqs'])
    if k == 'sgpr':
        model = (vfe_models if case['vfe'] else aep_models).SGPR(d['x'], d['y'], case['M'])
        mb = case['N']
    elif k == 'sgplvm':
        model = aep_models.SGPLVM(d['y'], case['Q'], case['M']).set_fused(case['fused'])
        mb = case['N']
    elif k == 'sgpssm':
        model = aep_models.SGPSSM(d['y'], case['Din'], case['M']).set_fused()
        mb = case['T']
    else:
        model = aep_models.SDGPR(d['x'], d['y'], case['M'], d['sizes'][1:-1]).set_fused()
        mb = case['N']
    if k == 'predict':
        model.update_hypers(p)
        return dict(kind=k, model=model, xs=d['xs'])
    if case['graph']:
        return dict(kind='graph', graph=graphs.GraphedObjective(model, p, mb, ALPHA))
    dp = aep_models.DeviceParams({n: np.shape(v) for n, v in p.items()})
    return dict(kind='eager', model=model, params=dp.upload(p), mb=mb)


def run(st):
    k = st['kind']
    if k == 'graph':
        return st['graph']()
    if k == 'eager':
        return st['model'].objective_function_device(st['params'], st['mb'], alpha=ALPHA)
    if k == 'predict':
        return st['model'].predict_f(st['xs'])
    if k == 'serve':
        return st['store'].predict_many(st['reqs'])
    from geepee_amd import autograd
    if not st['grad']:
        with torch.no_grad():
            return autograd.moment_match(*st['in'])
    out = autograd.moment_match(*st['in']) if k == 'mm' else autograd.psi_statistics(*st['in'])
    return list(out), list(torch.autograd.grad(out, st['in'], st['up']))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _mm_flops(N, M, Q, D, grad):
    """One moment-matched layer over N points: per unordered inducing pair the exponent's
    cross terms, an exp and the contraction; the adjoint's dpsi2, dBhat and moment sums."""
    pairs = N * M * (M + 1) / 2.0
    f = pairs * (2 * Q + 20 + 2 * D)
    return f + pairs * (2 * D + 2 * D + 4 * (Q + 1)) if grad else f


def _chain_flops(M, D, grad):
    """q(u) set-up of a layer: 1 + 2D inverses, the products of the predictive forms; adjoint."""
    f = (1 + 2 * D) * 1.0 * M ** 3 + 5.0 * D * M ** 3
    return f + 9.0 * D * M ** 3 + 6.0 * M ** 3 if grad else f


def _det_flops(N, M, Q, D, grad):
    f = N * M * (3.0 * Q + 20 + 2 * D) + 1.0 * N * M * M * D
    return f + 1.0 * N * M * M * D + N * M * (6.0 * Q + 4 * D) if grad else f


def _params(case):
    M, k = case['M'], case['kind']
    lay = lambda Din, Dout: M * Din + Din + 1 + Dout * (M * (M + 1) / 2 + M)
    if k == 'sgpr':
        return lay(case['Din'], case['Dout'])
    if k == 'sgplvm':
        return lay(case['Q'], case['D']) + 2 * case['N'] * case['Q']
    if k == 'sgpssm':
        return lay(case['Din'], case['Din']) + 2 * case['T'] * case['Din'] + case['Dout'] * (case['Din'] + 1)
    L = case.get('L', 2)
    return lay(case['Din'], case['H']) + (L - 2) * lay(case['H'], case['H']) + lay(case['H'], 1)


def work(case):
    k = case['kind']
    if k == 'sgpr':
        N, M, Q, D = case['N'], case['M'], case['Din'], case['Dout']
        return {'flops': _chain_flops(M, D, True) + _det_flops(N, M, Q, D, True),
                'bytes': 8 * (2 * _params(case) + N * (Q + D))}
    if k == 'sgplvm':
        N, M, Q, D = case['N'], case['M'], case['Q'], case['D']
        return {'flops': _chain_flops(M, D, True) + _mm_flops(N, M, Q, D, True),
                'bytes': 8 * (2 * _params(case) + N * D)}
    if k == 'sdgpr':
        N, M, H, L = case['N'], case['M'], case['H'], case['L']
        f = _chain_flops(M, H, True) + _det_flops(N, M, case['Din'], H, True)
        for i in range(1, L):
            D = H if i < L - 1 else 1
            f += _chain_flops(M, D, True) + _mm_flops(N, M, H, D, True)
        return {'flops': f, 'bytes': 8 * (2 * _params(case) + N * (case['Din'] + 1))}
    if k == 'sgpssm':
        T, M, Q, D = case['T'], case['M'], case['Din'], case['Dout']
        f = _chain_flops(M, Q, True) + _mm_flops(T, M, Q, Q, True) + T * (D ** 3 + 6.0 * D * D * Q)
        return {'flops': f, 'bytes': 8 * (2 * _params(case) + T * D)}
    if k == 'mm':
        N, M, Q, D = case['N'], case['M'], case['Q'], case['D']
        b = 2 * N * Q + M * Q + D * M + D * M * M + 2 * N * D
        return {'flops': _mm_flops(N, M, Q, D, case['grad']),
                'bytes': 8 * (2 * b + 2 * N * D if case['grad'] else b)}
    if k == 'psi':
        N, M, Q = case['N'], case['M'], case['Q']
        return {'flops': N * M * (M + 1) / 2.0 * (2 * Q + 20 + 2 + 4 * (Q + 1)),
                'bytes': 8 * (2 * N * M * M + 2 * N * M + 4 * N * Q + 2 * M * Q)}
    if k == 'predict':
        N, M, H = case['N'], case['M'], case['H']
        return {'flops': _det_flops(N, M, case['Din'], H, False) + _mm_flops(N, M, H, 1, False),
                'bytes': 8 * (N * (case['Din'] + 2) + (H + 1) * M * M)}
    f, b = _serve_work(case)
    return {'flops': f, 'bytes': 8 * b}


def _cost(case):
    w = work(case)
    return max(w['bytes'] / 4e12, w['flops'] / 4e13)


# ---------------------------------------------------------------------------
# plain torch in float64
# ---------------------------------------------------------------------------

def _dev():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


def _se(x, z, ls, sf):
    w = torch.exp(-ls)
    r = sum((x[:, q:q + 1] * w[q] - z[None, :, q] * w[q]) ** 2 for q in range(x.shape[1]))
    return torch.exp(2 * sf - 0.5 * r)


def _psi1(mx, vx, z, ls, sf):
    l = torch.exp(2 * ls)
    e = 0.0
    for q in range(mx.shape[1]):
        s = l[q] + vx[:, q:q + 1]
        e = e + 0.5 * torch.log(l[q] / s) - 0.5 * (mx[:, q:q + 1] - z[None, :, q]) ** 2 / s
    return torch.exp(2 * sf + e)


def _psi2(mx, vx, z, ls, sf):
    l = torch.exp(2 * ls)
    e = 0.0
    for q in range(mx.shape[1]):
        s = l[q] + 2 * vx[:, q, None, None]
        zq = z[:, q]
        h = 0.5 * (zq[:, None] + zq[None, :])
        e = e + 0.5 * torch.log(l[q] / s) - (mx[:, q, None, None] - h) ** 2 / s \
            - (zq[:, None] - zq[None, :]) ** 2 / (4 * l[q])
    return torch.exp(4 * sf + e)


def _match(mx, vx, z, ls, sf, A, B):
    """Moment-matched mean and variance, point blocks recomputed in the backward."""
    def block(m_, v_, *a):
        p1, p2 = _psi1(m_, v_, *a[:3]), _psi2(m_, v_, *a[:3])
        n = m_.shape[0]
        m = p1 @ a[3].T
        return m, torch.exp(2 * a[2]) + p2.reshape(n, -1) @ a[4].reshape(a[4].shape[0], -1).T - m ** 2
    step = max(1, int(1.2e7 / z.shape[0] ** 2))
    out = [checkpoint(block, mx[i:i + step], vx[i:i + step], z, ls, sf, A, B, use_reentrant=False)
           for i in range(0, mx.shape[0], step)]
    return torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out])


def _spd(A):
    """Inverse and log-determinant."""
    L = torch.linalg.cholesky(A)
    return torch.cholesky_inverse(L), 2 * torch.log(torch.diagonal(L, dim1=-2, dim2=-1)).sum(-1)


class _Exact(object):
    """One layer from its parameter dict (leaves on the CPU; M x M algebra there)."""

    def __init__(self, p, N, sfx=''):
        self.z, self.ls, self.sf = p['zu' + sfx], p['ls' + sfx], p['sf' + sfx]
        eta, self.th = p['eta1_R' + sfx], p['eta2' + sfx]
        self.N, (self.D, self.M) = N, self.th.shape
        i, j = np.triu_indices(self.M)
        i, j = torch.as_tensor(i), torch.as_tensor(j)
        R = torch.zeros(self.D, self.M, self.M, dtype=F64)
        R = R.index_put((torch.arange(self.D)[:, None], i[None], j[None]),
                        torch.where(i == j, torch.exp(eta), eta))
        self.t1 = R.transpose(1, 2) @ R
        self.K = _se(self.z, self.z, self.ls, self.sf) + JITTER * torch.eye(self.M, dtype=F64)
        self.Ki, self.ldK = _spd(self.K)

    def q(self, beta):
        S, ld = _spd(self.Ki + beta * self.t1)
        mu = beta * (S @ self.th[..., None])[..., 0]
        return S, mu, ld

    def forms(self, S, mu):
        A = mu @ self.Ki
        B = self.Ki @ S @ self.Ki - self.Ki
        return A, B, B + A[:, :, None] * A[:, None, :]

    def cavity(self, alpha):
        """Predictive forms of the cavity and phi."""
        N = self.N
        beta = (N - alpha) / N
        S, mu, ld = self.q(1.0)
        Sh, muh, ldh = self.q(beta)
        p = 0.5 * ((mu * self.th).sum() - ld.sum())
        c = 0.5 * (beta * (muh * self.th).sum() - ldh.sum())
        phi = self.D * 0.5 * self.ldK + (N / alpha - 1.0) * p - N / alpha * c
        return self.forms(Sh, muh), phi

    def hyp(self, dev):
        return self.z.to(dev), self.ls.to(dev), self.sf.to(dev)

    def det(self, x, A, B):
        dev = x.device
        z, ls, sf = self.hyp(dev)
        k = _se(x, z, ls, sf)
        A, B = A.to(dev), B.to(dev)
        v = torch.stack([((k @ B[d]) * k).sum(1) for d in range(B.shape[0])], 1)
        return k @ A.T, torch.exp(2 * sf) + v

    def match(self, m, v, A, B):
        dev = m.device
        return _match(m, v, *self.hyp(dev), A.to(dev), B.to(dev))


def _gauss(m, v, y, sn, alpha):
    s2 = torch.exp(2 * sn)
    vt = v + s2 / alpha
    lz = -0.5 * (torch.log(2 * math.pi * vt) + (y - m) ** 2 / vt)
    n = m.numel()
    return lz.sum() + n * (0.5 * torch.log(2 * math.pi * s2 / alpha) - 0.5 * alpha * torch.log(2 * math.pi * s2))


def _energy(case, d, p, dev):
    k, a = case['kind'], ALPHA
    y = torch.as_tensor(d['y'], device=dev)
    N = y.shape[0]
    if k == 'sgpr':
        x = torch.as_tensor(d['x'], device=dev)
        L = _Exact(p, N)
        sn = p['sn'].to(dev)
        if case['vfe']:
            S, mu, ld = L.q(1.0)
            A, B, _ = L.forms(S, mu)
            m, v = L.det(x, A, B)
            s2 = torch.exp(2 * sn)
            lik = (-0.5 * torch.log(2 * math.pi * s2) - 0.5 * ((y - m) ** 2 + v) / s2).sum()
            kl = 0.5 * ((L.Ki * (S + mu[:, :, None] * mu[:, None, :])).sum() - L.D * L.M
                        + L.D * L.ldK + ld.sum())
            return (kl - lik.cpu()) / N
        (A, B, _), phi = L.cavity(a)
        m, v = L.det(x, A, B)
        return (phi - _gauss(m, v, y, sn, a).cpu() / a) / N
    if k == 'sdgpr':
        x = torch.as_tensor(d['x'], device=dev)
        e, m, v = 0.0, None, None
        for i in range(case['L']):
            L = _Exact(p, N, '_%d' % i)
            (A, B, Bs), phi = L.cavity(a)
            e = e + phi
            m, v = L.det(x, A, B) if i == 0 else L.match(m, v, A, Bs)
        return (e - _gauss(m, v, y, p['sn'].to(dev), a).cpu() / a) / N
    if k == 'sgplvm':
        L = _Exact(p, N)
        (A, _, Bs), phi = L.cavity(a)
        t1, t2 = p['x1'], torch.exp(2 * p['x2'])
        c1, c2, p1, p2 = (1 - a) * t1, 1 + (1 - a) * t2, t1, 1 + t2
        m, v = L.match((c1 / c2).to(dev), (1 / c2).to(dev), A, Bs)
        ph = lambda u, w: 0.5 * (u ** 2 / w - torch.log(w)).sum()
        x = -ph(c1, c2) / a - (1.0 - 1.0 / a) * ph(p1, p2)
        return phi + x - _gauss(m, v, y, p['sn'].to(dev), a).cpu() / a
    L = _Exact(p, N - 1, '_dynamic')
    (A, _, Bs), phi = L.cavity(a)
    f1, f2 = p['x_factor_1'].to(dev), torch.exp(2 * p['x_factor_2'].to(dev))
    w = torch.full((N, 1), 3.0, dtype=F64, device=dev)
    w[0] = w[-1] = 2.0
    pr = torch.zeros(N, 1, dtype=F64, device=dev)
    pr[0] = 1.0
    p1, p2 = w * f1, w * f2 + pr
    c1, c2 = p1 - a * f1, p2 - a * f2
    cm, cv = c1 / c2, 1 / c2
    m, v = L.match(cm[:-1], cv[:-1], A, Bs)
    s2 = torch.exp(2 * p['sn'].to(dev))
    vs, md = cv[1:] + v + s2 / a, cm[1:] - m
    dyn = (-0.5 * md ** 2 / vs - 0.5 * torch.log(1 + a * (cv[1:] + v) / s2)
           - 0.5 * a * torch.log(2 * math.pi * s2)).sum()
    C, R = p['C_emission'].to(dev), torch.exp(2 * p['R_emission'].to(dev))
    Vy = torch.diag(R / a)[None] + torch.einsum('ac,nc,bc->nab', C, cv, C)
    Lc = torch.linalg.cholesky(Vy)
    u = torch.linalg.solve_triangular(Lc, (y - cm @ C.T)[..., None], upper=False)[..., 0]
    D = y.shape[1]
    emi = -0.5 * (u ** 2).sum() - torch.log(torch.diagonal(Lc, dim1=1, dim2=2)).sum() \
        + N * (0.5 * torch.log(R / a).sum() - 0.5 * D * a * math.log(2 * math.pi) - 0.5 * a * torch.log(R).sum())
    g = torch.full((N, 1), -(1 - 1 / a), dtype=F64, device=dev)
    h = torch.full((N, 1), -1 / a, dtype=F64, device=dev)
    g[:-1] += 1 / a
    g[1:] += 1 / a
    h[:-1] -= 1 / a
    h[1:] -= 1 / a
    ph = lambda u_, w_: 0.5 * (u_ ** 2 / w_ - torch.log(w_))
    xc = (g * ph(p1, p2) + h * ph(c1, c2)).sum()
    return (phi + (xc - (dyn + emi) / a).cpu()) / N


def _predict(p, N, sizes, xs, dev, sfx=True):
    x = torch.as_tensor(xs, device=dev)
    m = v = None
    with torch.no_grad():
        for i in range(len(sizes) - 1):
            L = _Exact(p, N, '_%d' % i if sfx else '')
            S, mu, _ = L.q(1.0)
            A, B, Bs = L.forms(S, mu)
            m, v = L.det(x, A, B) if i == 0 else L.match(m, v, A, Bs)
    return m, v


def exact(case, seed):
    d, p = _inputs(case, seed)
    k, dev = case['kind'], _dev()
    if k in ('mm', 'psi'):
        t = {n: torch.as_tensor(v, device=dev) for n, v in d.items()}
        names = ['mx', 'vx', 'z', 'ls', 'sf'] + (['A', 'B'] if k == 'mm' else [])
        grad = k == 'psi' or case['grad']
        ins = [t[n].requires_grad_(grad) for n in names]
        if not grad:
            with torch.no_grad():
                return _match(*ins)
        if k == 'mm':
            out, up = _match(*ins), [t['gm'], t['gv']]
        else:
            out = _psi1(*ins), _psi2(*ins)
            up = [t['g1'], torch.einsum('nd,dab->nab', t['g2'], t['B2'])]
        g = torch.autograd.grad(out, ins, up)
        return [o.detach() for o in out], list(g)
    if k == 'serve':
        out, keep = [], {}
        for i, X in d['reqs']:
            s = d['models'][i]
            q = {n: torch.as_tensor(v) for n, v in s['params'].items()}
            m, v = _predict(q, s['N'], [s['Din']] + s['hidden'] + [1], X, dev, s['kind'] != 'sgpr')
            out.append((m, v))
        return out
    q = {n: torch.as_tensor(v).requires_grad_(k != 'predict') for n, v in p.items()}
    if k == 'predict':
        return _predict(q, 4 * case['M'], d['sizes'], d['xs'], dev)
    e = _energy(case, d, q, dev)
    names = sorted(q)
    g = torch.autograd.grad(e.reshape(()), [q[n] for n in names])
    return torch.cat([e.detach().reshape(1).to(dev)] + [x.reshape(-1).to(dev) for x in g])
