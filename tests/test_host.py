"""Host-side logic that needs no GPU: launch plans, the autotuner cache, request
generation."""
import json

import numpy as np
import pytest

from geepee_amd import autotune, dops
from geepee_amd.serving import make_requests


def _ntiles(M):
    T = (M + 15) // 16
    return T * (T + 1) // 2


@pytest.mark.parametrize('N', [1, 15, 16, 17, 1000, 4096, 20000])
@pytest.mark.parametrize('M', [1, 16, 33, 100, 128, 200, 256])
def test_fused_plan_within_kernel_limits(N, M, monkeypatch, tmp_path):
    monkeypatch.setenv('GEEPEE_AMD_TUNE_CACHE', str(tmp_path / 'none.json'))
    autotune.clear()
    p = dops.fused_plan(N, M, 4, 8)
    assert p['nsub'] in (1, 2, 4)
    assert 1 <= p['splits_f'] <= _ntiles(M)
    assert 1 <= p['splits_b'] <= (M + 15) // 16
    assert 1 <= p['nsplit'] <= -(-N // 16)


@pytest.mark.parametrize('N,M', [(16, 16), (1000, 100), (4096, 128), (10000, 200)])
def test_fused_candidates_within_kernel_limits(N, M):
    fwd, bpt, bpr = autotune.fused_candidates(N, M)
    assert fwd and bpt and bpr
    for c in fwd:
        assert c['nsub'] in (1, 2, 4) and 1 <= c['splits_f'] <= _ntiles(M)
    assert all(1 <= s <= (M + 15) // 16 for s in bpt)
    assert all(1 <= s <= -(-N // 16) for s in bpr)


def test_gemm_candidates():
    c = autotune.gemm_candidates(128, 128, 4096, 1)
    assert {'tile': 64, 'splits': 1} in c and {'tile': 32, 'splits': 1} in c
    assert all(4096 // x['splits'] >= 64 for x in c)


def test_autotune_cache_round_trip(monkeypatch, tmp_path):
    path = tmp_path / 'tune.json'
    monkeypatch.setenv('GEEPEE_AMD_TUNE_CACHE', str(path))
    autotune.clear()
    assert autotune.lookup('fused', (100, 20, 3, 4)) is None
    plan = {'nsub': 2, 'splits_f': 3, 'splits_b': 5, 'nsplit': 7}
    autotune.store('fused', (100, 20, 3, 4), plan)
    assert json.loads(path.read_text())
    autotune.clear()
    assert autotune.lookup('fused', (100, 20, 3, 4)) == plan
    assert dops.fused_plan(100, 20, 3, 4) == plan
    assert dops.fused_plan(100, 20, 3, 4, tuned=False) != plan
    autotune.clear()


def test_make_requests_shape():
    reqs = make_requests(8, 500, 1000.0, [1 + i for i in range(8)], seed=3)
    t = np.array([r[0] for r in reqs])
    assert np.all(np.diff(t) >= 0)
    assert abs(len(reqs) / t[-1] - 1000.0) < 200.0
    for _, mid, X in reqs:
        assert 0 <= mid < 8 and X.shape[1] == 1 + mid and 1 <= X.shape[0] <= 4096


def _unpack_R(eta, M):
    R = np.zeros((M, M))
    R[np.triu_indices(M)] = eta
    R[np.diag_indices(M)] = np.exp(np.diag(R))
    return R


def test_layer_init_matches_reference_recipe():
    """base_models.py:518-597: kmeans2 on x, median-distance lengthscales, sf = log 0.5,
    theta1 = diag(1 / (0.5 U)) packed as an upper Cholesky factor with log diagonal,
    theta2 = theta1 linspace(-1, 1); the draws come from the global legacy RNG."""
    from geepee_amd import init
    from scipy.cluster.vq import kmeans2
    from scipy.spatial.distance import cdist
    rs = np.random.RandomState(0)
    x = rs.randn(40, 3)
    np.random.seed(5)
    p = init.sgp_layer(40, 7, 3, 2, True, x_train=x, key_suffix='_0')
    np.random.seed(5)
    zu, _ = kmeans2(x, 7, minit='points')
    alphas = [0.5 * np.random.rand(7) for _ in range(2)]
    assert np.array_equal(p['zu_0'], zu)
    d = cdist(x, x)
    assert np.allclose(p['ls_0'], np.log(np.median(d[np.triu_indices(40)]) / 2))
    assert np.allclose(p['sf_0'], np.log(0.5))
    for dd in range(2):
        R = _unpack_R(p['eta1_R_0'][dd], 7)
        assert np.allclose(R.T.dot(R), np.diag(1 / alphas[dd]))
        assert np.allclose(p['eta2_0'][dd], np.linspace(-1, 1, 7) / alphas[dd])
    np.random.seed(5)
    q = init.sgp_layer(40, 7, 3, 2, True, x_train=x, key_suffix='_0')
    assert all(np.array_equal(p[k], q[k]) for k in p)


def test_optimal_qu_is_the_collapsed_optimum():
    """Sigma = Kuu (Kuu + Kuf Kfu / sn2)^-1 Kuu and mu = Sigma Kuu^-1 Kuf y / sn2 (the
    optimum of the collapsed bound), in both parameterisations."""
    from geepee_amd import init
    rs = np.random.RandomState(1)
    x, y = rs.randn(30, 2), rs.randn(30, 2)
    np.random.seed(0)
    base = init.sgp_layer(30, 6, 2, 2, True, x_train=x)
    sn = np.log(0.3)
    Kuu = init._se(base['ls'], base['sf'], base['zu'], base['zu']) + 1e-5 * np.eye(6)
    Kfu = init._se(base['ls'], base['sf'], x, base['zu'])
    S = Kuu.dot(np.linalg.solve(Kuu + Kfu.T.dot(Kfu) / np.exp(2 * sn), Kuu))
    mu = S.dot(np.linalg.solve(Kuu, Kfu.T.dot(y))) / np.exp(2 * sn)
    for nat in (True, False):
        p = init.optimal_qu(dict(base), '', x, y, 6, nat, sn)
        for d in range(2):
            R = _unpack_R(p['eta1_R'][d], 6)
            t1 = R.T.dot(R)
            if nat:
                Sig = np.linalg.inv(np.linalg.inv(Kuu) + t1)
                m = Sig.dot(p['eta2'][d])
            else:
                Sig, m = t1, p['eta2'][d]
            assert np.allclose(Sig, S, rtol=1e-6, atol=1e-9)
            assert np.allclose(m, mu[:, d], rtol=1e-6, atol=1e-9)


def test_model_init_keys_and_shapes():
    from geepee_amd import init, workloads as W
    y, want = W.sgplvm_problem(N=60, Q=3, D=5, M=8, seed=2)
    np.random.seed(0)
    got = init.sgplvm(y, 3, 8)
    assert sorted(got) == sorted(want)
    assert all(np.shape(got[k]) == np.shape(want[k]) for k in want)
    y, want = W.sgpssm_problem(T=80, Din=2, Dout=3, M=6, seed=3)
    np.random.seed(0)
    got = init.sgpssm(y, 2, 6)
    assert sorted(got) == sorted(want)
    assert all(np.shape(got[k]) == np.shape(want[k]) for k in want)
    # the PCA projection is the reference's: leading eigenvectors of cov(y)
    P = init.pca_reduce(y, 2)
    w, V = np.linalg.eigh(np.cov(y.T))
    assert np.allclose(np.abs(P), np.abs((y - y.mean(0)).dot(V[:, ::-1][:, :2])))


def test_admission_respects_the_budget():
    from geepee_amd.serving import admit
    # fits: three requests of 100 bytes under a 350-byte budget
    assert admit([(100, 1), (100, 1), (100, 1), (100, 1)], 0, 350, 1 << 16, idle=True) == 3
    # the point cap stops a launch as the byte budget does
    assert admit([(10, 40), (10, 40)], 0, 1000, 64, idle=True) == 1
    # in-flight bytes count: the head waits while another launch holds the memory
    assert admit([(100, 1)], 300, 350, 1 << 16, idle=False) == 0
    # a request larger than the whole budget waits while anything is in flight ...
    assert admit([(500, 1), (10, 1)], 100, 350, 1 << 16, idle=False) == 0
    assert admit([(500, 1)], 0, 350, 1 << 16, idle=False) == 0
    # ... and then runs alone
    assert admit([(500, 1), (10, 1)], 0, 350, 1 << 16, idle=True) == 1
    # the queue is read only as far as the launch reaches
    seen = []

    def sizes():
        for i in range(10):
            seen.append(i)
            yield (100, 1)
    assert admit(sizes(), 0, 250, 1 << 16, idle=True) == 2
    assert seen == [0, 1, 2]


def test_spd_status_raises_linalg_error():
    """check_status reads the device status pair written by gpx_status_fold: entry 0 is
    the last evaluation's largest info (k+1 for a failed pivot k), entry 1 the sticky
    flag of the optimiser loop."""
    import types
    import torch
    from geepee_amd.aep_models import Base_Model
    m = types.SimpleNamespace(_status=torch.tensor([0, 0], dtype=torch.int32))
    Base_Model.check_status(m)
    Base_Model.check_status(m, sticky=True)
    m._status = torch.tensor([4, 4], dtype=torch.int32)
    with pytest.raises(np.linalg.LinAlgError, match='pivot 3'):
        Base_Model.check_status(m)
    m._status = torch.tensor([0, 2], dtype=torch.int32)
    Base_Model.check_status(m)
    with pytest.raises(np.linalg.LinAlgError, match='during optimisation'):
        Base_Model.check_status(m, sticky=True)


def _stub_layer(monkeypatch, M=20, Q=3, D=2):
    """A layer on the CPU whose kernels are stand-ins that count the operand's formations."""
    import torch
    from geepee_amd import layers
    formed = []
    monkeypatch.setattr(layers.dops, 'sym_pairmajor', lambda B: formed.append(B) or B.permute(1, 2, 0))
    monkeypatch.setattr(layers.dops, 'fused_mm_fwd', lambda *a, **k: (None, a[6], a[6]))
    monkeypatch.setattr(layers, 'mm', lambda A, B, *a, **k: A)
    monkeypatch.setattr(layers, '_sandwich', lambda A, B, C, **k: B)
    L = layers.SGP_Layer(100, Q, D, M)
    L.zu, L.ls, L.sf = torch.zeros(M, Q), torch.zeros(Q), torch.zeros(1)
    L.Kuuinv, L.mu, L.Su, L.Splusmm = torch.zeros(M, M), torch.zeros(D, M), *torch.zeros(2, D, M, M)
    return L, formed


def test_gaussian_operand_comes_with_the_posterior(monkeypatch):
    """The fused layout of B_sto is formed together with A, B_sto and B_det, so whatever orders
    those for another stream orders it as well."""
    import torch
    x = torch.zeros(5, 3)
    L, formed = _stub_layer(monkeypatch)
    L.forward_prop_thru_post(x, x)
    L.forward_prop_thru_post(x, x)
    assert len(formed) == 1 and L._Bp_post is not None
    L, formed = _stub_layer(monkeypatch)
    L._posterior_predictive(gaussian=False)
    assert not formed and L._Bp_post is None
    L._pred_ready = False
    L._posterior_predictive(gaussian=True)
    assert len(formed) == 1 and L._Bp_post is not None
    L, formed = _stub_layer(monkeypatch, Q=16)     # outside the fused kernels
    L._posterior_predictive(gaussian=True)
    assert not formed and L._Bp_post is None


def test_gaussian_operand_formed_by_a_call_is_not_kept(monkeypatch):
    """On a posterior formed without it (by a deterministic call, say on another stream), a call
    forms its own operand and leaves nothing behind for callers that could not wait for it."""
    import torch
    x = torch.zeros(5, 3)
    L, formed = _stub_layer(monkeypatch)
    L._posterior_predictive()
    L.forward_prop_thru_post(x, x)
    L.forward_prop_thru_post(x, x)
    assert len(formed) == 2 and L._Bp_post is None


@pytest.mark.parametrize('N,M,D', [(20000, 128, 32), (50000, 100, 32), (100000, 256, 32), (130000, 16, 32),
                                   (1000000, 64, 4), (4096, 128, 32)])
def test_noalloc_plan_fits_the_scratch(N, M, D, monkeypatch, tmp_path):
    """The allocation-free forward takes every shape whose partial sums fit the scratch at one
    split, however many splits the plan would like."""
    from geepee_amd import _lib
    monkeypatch.setenv('GEEPEE_AMD_TUNE_CACHE', str(tmp_path / 'none.json'))
    autotune.clear()
    seen = []
    monkeypatch.setattr(dops, 'call', lambda name, *a: seen.append((name,) + a))
    monkeypatch.setattr(dops, 'P', lambda t: t)
    monkeypatch.setattr(dops, 'S', lambda: 0)
    shape = lambda *s: type('T', (), {'shape': s})()
    dops.fused_mm_fwd_noalloc(shape(N, 3), shape(N, 3), shape(M, 3), None, None, shape(D, M), None, None, None, None)
    (name, splits), = [(c[0], c[12]) for c in seen]
    assert name == 'gpx_fused_mm_fwd_noalloc' and splits >= 1
    assert _lib.query('gpx_fused_fwd_workspace', N, M, D, splits) <= _lib.query('gpx_fused_fwd_noalloc_max')
    autotune.clear()


@pytest.mark.parametrize('kind,shape,plan', [
    ('fused', (500, 40, 3, 4), {'nsub': 4, 'splits_f': 6, 'splits_b': 3, 'nsplit': 1}),
    ('gemm', (128, 128, 4096, 1, 1, 0), {'splits': 64, 'tile': 64})])
def test_plans_of_other_kernels_are_not_read(kind, shape, plan, monkeypatch, tmp_path):
    """A cache file from before the kernels' knobs changed (keys without a revision) leaves the rules
    in place; it is kept when a new plan is stored beside it."""
    path = tmp_path / 'tune.json'
    old = 'gfx950|%s|%s' % (kind, ','.join(str(s) for s in shape))
    path.write_text(json.dumps({old: plan}))
    monkeypatch.setenv('GEEPEE_AMD_TUNE_CACHE', str(path))
    monkeypatch.setattr(autotune, '_tag', 'gfx950')
    autotune.clear()
    assert autotune.lookup(kind, shape) is None
    if kind == 'fused':
        assert dops.fused_plan(*shape) == dops.fused_plan(*shape, tuned=False)
    autotune.store(kind, shape, dict(plan, ms=1.0))
    autotune.clear()
    assert autotune.lookup(kind, shape) == dict(plan, ms=1.0)
    assert json.loads(path.read_text())[old] == plan
    autotune.clear()


def test_tuned_product_plan_not_used_with_a_tail(monkeypatch, tmp_path):
    """A plan is timed without the outer product and the second output; a product with either keeps
    the rule's split count and tile."""
    import torch
    monkeypatch.setenv('GEEPEE_AMD_TUNE_CACHE', str(tmp_path / 'tune.json'))
    autotune.clear()
    autotune.store('gemm', (20, 20, 2048, 1, 0, 0), {'splits': 3, 'tile': 64})
    seen = []
    monkeypatch.setattr(dops._lib, 'mm', lambda *a, **k: seen.append((k['splits'], k['tile'])))
    A, B, C, U = torch.zeros(20, 2048), torch.zeros(2048, 20), torch.zeros(20, 20), torch.zeros(1, 20)
    dops.mm(A, B, C)
    dops.mm(A, B, C, outer=(U, U, 1.0))
    dops.mm(A, B, C, second=(C, 1.0, None))
    assert seen == [(3, 64), (4, 0), (4, 0)]
    autotune.clear()


@pytest.mark.parametrize('N', [1, 10, 50, 100, 200, 600, 1000, 3001, 4096, 8000, 9999, 50000, 200000])
@pytest.mark.parametrize('M', [5, 16, 32, 48, 64, 100, 128, 200, 256])
def test_fused_plan_leaves_no_cu_idle(N, M):
    """Workgroups are not held back below the 256 CUs while there is work to split: the forward's
    tiles for few points, the adjoint's point ranges for few tiles (down to two blocks a range, or
    the 4 sqrt(blocks) at which summing the ranges' partials costs more than shorter ranges give)."""
    p = dops.fused_plan(N, M, 4, 8, tuned=False)
    nt, nb = _ntiles(M), -(-N // 16)
    blocks = -(-N // (16 * p['nsub']))
    if blocks <= 25 and nt > 8:
        assert blocks * p['splits_f'] >= 128 or p['splits_f'] == nt
    each = -(-nb // p['nsplit'])
    assert nt * p['nsplit'] >= 128 or each <= 3 or p['nsplit'] >= 0.8 * 4 * nb ** 0.5
    assert p['nsplit'] <= max(32, 4 * nb ** 0.5)
