"""GPU variogram estimation and fit against the CPU oracle.

Bins: pair counts exact, mean distances and estimator values 1e-12
relative.  Fits: differential evolution is stochastic (unseeded in the
reference), so a fit is compared by its objective on bounds that contain
the optimum: the GPU objective must be within 1e-3 of SciPy's (or below).
"""
import numpy as np
import pytest

from oracle import vgfit_oracle as V

pytestmark = pytest.mark.gpu


def _field(seed, n=260, n_act=200, r=25e3, model='Exp'):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0, 2e5, n)
    y = rng.uniform(0, 2e5, n)
    d = np.hypot(x[:, None] - x[None], y[:, None] - y[None])
    if model == 'Exp':
        c = np.exp(-3 * d / r)
    else:
        c = np.exp(-3 * (d / r) ** 2)
    c += 1e-6 * np.eye(n)
    z = np.linalg.cholesky(c) @ rng.standard_normal(n) * 2.0 + 5.0
    z[rng.choice(n, n - n_act, replace=False)] = np.nan
    return x, y, z


@pytest.mark.parametrize('evg', ['robust', 'classic'])
@pytest.mark.parametrize('mdr', [0.5, 0.7])
def test_bins_match_oracle(gpu, evg, mdr):
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    fields = [_field(s) for s in range(3)]
    x, y = fields[0][0], fields[0][1]
    rng = np.random.default_rng(9)
    vals = np.stack([_field(s)[2] for s in range(3)])
    f = BatchVariogramFitter(x, y)
    bh, bg, bn, nb = f.empirical(vals, mdr, 50, evg)
    for t in range(3):
        ok = ~np.isnan(vals[t])
        ref = V.empirical(x[ok], y[ok], vals[t][ok], mdr, 50, evg)
        k = int(nb[t])
        assert k == ref.shape[0]
        np.testing.assert_array_equal(bn[t, :k].cpu().numpy(), ref[:, 2])
        np.testing.assert_allclose(bh[t, :k].cpu().numpy(), ref[:, 0],
                                   rtol=1e-12)
        np.testing.assert_allclose(bg[t, :k].cpu().numpy(), ref[:, 1],
                                   rtol=1e-12)


def test_de_objective_matches_scipy(gpu):
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    x, y, _ = _field(0)
    vals = np.stack([_field(s)[2] for s in (0, 1)] +
                    [_field(s, model='Gau', r=40e3)[2] for s in (2, 3)])
    f = BatchVariogramFitter(x, y)
    kw = dict(mdr=0.5, nk=50, perm_r_list=[1, 2], fit_vgs=['Sph', 'Exp'],
              fil_nug_vg='Nug', range_ub=2e5)
    out, det = f.fit(vals, seed=5, return_details=True, **kw)
    cands = det['cands']
    for k, t in enumerate(det['steps']):
        ok = ~np.isnan(vals[t])
        strs, ref = V.fit(x[ok], y[ok], vals[t][ok], seed=11, **kw)
        for c, o in enumerate(cands):
            fg = det['fun'][k, c]
            fc = ref['funs'][o][0]
            assert fg <= fc * (1 + 1e-3) + 1e-12, (t, o, fg, fc)
        assert out[t] is not None and len(out[t]) == 1


def test_de_candidates_independent_of_launch_lds(gpu):
    """Each (step, candidate) DE is one workgroup whose LDS is sized for the
    largest candidate of its launch: one-component candidates give the same
    bits alone (rows of 2 parameters, 200 members) and beside three- and
    four-component ones (rows of 8, 800 members: 800 x 8 x 2 doubles, 100 KiB
    of LDS per workgroup), and
    every candidate's objective is the oracle's objective at its
    parameters."""
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    x, y, _ = _field(0)
    vals = np.stack([_field(s)[2] for s in (0, 1)])
    f = BatchVariogramFitter(x, y)
    # four model types: permutations of up to 4 components (the size is
    # capped at the number of types, fitvgs.py's candidate rule)
    kw = dict(mdr=0.5, nk=50, fit_vgs=['Sph', 'Exp', 'Lin', 'Gau'],
              fil_nug_vg='Nug', range_ub=2e5, opt_iters=300, seed=3,
              return_details=True)
    _, d1 = f.fit(vals, perm_r_list=[1], **kw)
    _, d4 = f.fit(vals, perm_r_list=[1, 3, 4], **kw)
    n1 = len(d1['cands'])
    assert list(d4['cands'][:n1]) == list(d1['cands'])
    assert max(len(o) for o in d4['cands']) == 4
    np.testing.assert_array_equal(d4['params'][:, :n1], d1['params'])
    np.testing.assert_array_equal(d4['fun'][:, :n1], d1['fun'])
    np.testing.assert_array_equal(d4['nit'][:, :n1], d1['nit'])
    bh = d4['bins'][0].cpu().numpy()
    bg = d4['bins'][1].cpu().numpy()
    nb = d4['bins'][3].cpu().numpy()
    for k in range(len(d4['steps'])):
        h, g = bh[k, :nb[k]], bg[k, :nb[k]]
        for c, o in enumerate(d4['cands']):
            p = d4['params'][k, c, :2 * len(o)]
            assert np.all(d4['params'][k, c, 2 * len(o):] == 0.0)
            ref = V.objective(p, list(o), h, g)
            np.testing.assert_allclose(d4['fun'][k, c], ref, rtol=1e-9)


def test_fit_strings_parse_and_skip_rules(gpu):
    from spinterps_amd import _lib
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    x, y, z = _field(4)
    vals = np.stack([z, np.full_like(z, np.nan), np.where(np.isnan(z), z, 3.0)])
    f = BatchVariogramFitter(x, y)
    out = f.fit(vals, mdr=0.7, perm_r_list=[1, 2], fit_vgs=['Sph', 'Exp'],
                fil_nug_vg='Nug', seed=1, opt_iters=2000)
    assert out[1] is None            # no values
    assert out[2] is None            # no spread (fitvgs.py:176-180)
    v = _lib.parse_vg(out[0][0])
    assert 1 <= v.n <= 2


def test_fit_choice_and_strings_match_oracle(gpu):
    """The AIC choice, range sorting, skips and output strings
    (vgs.py:771-846) of the GPU fit against the oracle's select_models and
    vg_strings fed with the GPU's own optimised objectives and parameters
    (DE itself is stochastic; its objectives are checked against SciPy
    above): the strings must be identical, for one and for two kept
    models."""
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    x, y, _ = _field(0)
    vals = np.stack([_field(5, model='Gau', r=60e3)[2], _field(6, r=20e3)[2],
                     _field(7, model='Gau', r=30e3)[2]])
    f = BatchVariogramFitter(x, y)
    for n_best in (1, 2):
        kw = dict(mdr=0.5, nk=50, perm_r_list=[1, 2],
                  fit_vgs=['Sph', 'Exp', 'Gau'], fil_nug_vg='Nug',
                  range_ub=2e5, n_best=n_best)
        out, det = f.fit(vals, seed=3, return_details=True, **kw)
        cands = det['cands']
        for k, t in enumerate(det['steps']):
            n = int((~np.isnan(vals[t])).sum())

            def solve(o, k=k):
                c = cands.index(o)
                return det['fun'][k, c], det['params'][k, c, :2 * len(o)]
            best, _, _ = V.select_models(cands, solve, n, 0.01, n_best)
            assert out[t] == V.vg_strings(best)[::-1], (t, out[t])


def test_de_three_component_objective_matches_scipy(gpu):
    """A three-component candidate (six parameters) where SciPy evolves
    50 x 6 x 6 = 1800 members and the GPU at most 800: the GPU objective is
    within 1e-3 of SciPy's."""
    from scipy.optimize import differential_evolution
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    x, y, _ = _field(0)
    vals = _field(8, r=30e3)[2][None, :]
    f = BatchVariogramFitter(x, y)
    kw = dict(mdr=0.5, nk=50, perm_r_list=[3], fit_vgs=['Sph', 'Exp', 'Gau'],
              fil_nug_vg='Nug', range_ub=2e5)
    _, det = f.fit(vals, seed=5, return_details=True, **kw)
    cands = det['cands']
    o = ('Nug', 'Exp', 'Gau')
    c = cands.index(o)
    ok = ~np.isnan(vals[0])
    z = vals[0][ok]
    bins = V.empirical(x[ok], y[ok], z, 0.5, 50, 'robust')
    h, g = bins[:, 0], bins[:, 1]
    bnds = V.bounds_for(o, h[0], g[0], np.var(z), 'Nug', 2e5)
    assert len(bnds) == 6
    res = differential_evolution(V.objective, bnds, args=(o, h, g, None),
                                 maxiter=10000, popsize=len(bnds) * 50,
                                 polish=False, seed=np.random.default_rng(2))
    fg = det['fun'][0, c]
    assert fg <= res.fun * (1 + 1e-3) + 1e-12, (fg, res.fun)


@pytest.mark.parametrize('n,nk', [(24, 50), (130, 10), (400, 7)])
def test_de_every_model_and_bin_count(gpu, n, nk):
    """The device-wide evolution sums an energy in parts of max(64,
    bins / 16) bins (fewer than 64 bins, a few parts, 16 ragged parts) with
    loops of its own for Nug, Sph, Exp and Gau: every candidate's objective
    is the oracle's at its parameters, and a step gives the same bits alone
    as among others."""
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0, 2e5, n), rng.uniform(0, 2e5, n)
    vals = rng.gamma(2.0, 3.0, (3, n))
    vals[1, rng.choice(n, n // 3, replace=False)] = np.nan
    f = BatchVariogramFitter(x, y)
    kw = dict(mdr=0.5, nk=nk, perm_r_list=[1, 2], fit_vgs=['all'],
              fil_nug_vg='Nug', range_ub=2e5, opt_iters=60, seed=3,
              return_details=True)
    _, det = f.fit(vals, **kw)
    _, one = f.fit(vals[:1], **kw)
    np.testing.assert_array_equal(one['params'][0], det['params'][0])
    np.testing.assert_array_equal(one['nit'][0], det['nit'][0])
    bh, bg, nb = (det['bins'][k].cpu().numpy() for k in (0, 1, 3))
    for k in range(3):
        h, g = bh[k, :nb[k]], bg[k, :nb[k]]
        for c, o in enumerate(det['cands']):
            p = det['params'][k, c, :2 * len(o)]
            ref = V.objective(p, list(o), h, g)
            # a residual carries some 16 roundings of the size of g, which
            # is what is left where few bins are fitted almost exactly:
            # d(sum r^2) <= 2 sqrt(sum r^2) sqrt(sum (16 u g)^2)
            np.testing.assert_allclose(
                det['fun'][k, c], ref, rtol=1e-9,
                atol=2 * np.sqrt(ref) * 16 * 1.2e-16 * np.linalg.norm(g))


def test_de_captured_matches_eager(gpu):
    """A captured launch cannot be followed by the host's reads and evolves
    each candidate in one workgroup: the same random streams, so the same
    generations, and objectives equal to the order of the energy sums."""
    import ctypes
    import torch
    from spinterps_amd import _lib
    from spinterps_amd.variograms.fitvgs import (TYPE_ID, BatchVariogramFitter,
                                                 candidate_sets)
    x, y, _ = _field(0)
    vals = np.stack([_field(s)[2] for s in (0, 1)])
    f = BatchVariogramFitter(x, y)
    bh, _, _, nb = bins = f.empirical(vals)
    cands = candidate_sets(['Sph', 'Exp', 'Gau'], [1, 2], 'Nug')
    var = np.nanvar(vals, axis=1)
    _, fun, nit = f.de(bins, var, cands, 'Nug', seed=4, range_ub=2e5)
    spec = np.zeros((len(cands), 6), np.int32)
    for c, o in enumerate(cands):
        spec[c, 0] = len(o)
        spec[c, 1:1 + len(o)] = [TYPE_ID[m] for m in o]
        spec[c, 5] = 1 if len(o) > 1 and o[0] == 'Nug' else 0
    ctx, st = _lib.Context(0), torch.cuda.Stream()
    ctx.set_stream(st.cuda_stream)
    vd = torch.as_tensor(var, device='cuda')
    par2 = torch.zeros((2, len(cands), 8), dtype=torch.float64, device='cuda')
    fun2, nit2 = torch.zeros_like(fun), torch.zeros_like(nit)

    def call():
        _lib.check(_lib.lib().spk_vgfit_de_dev(
            ctx.h, bh.data_ptr(), bins[1].data_ptr(), nb.data_ptr(),
            bh.shape[1], vd.data_ptr(), 2,
            spec.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), len(cands),
            10000, 50, 0.01, 2e5, 4, par2.data_ptr(), fun2.data_ptr(),
            nit2.data_ptr()))
    torch.cuda.synchronize()
    call()  # sizes the context's scratch
    st.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        call()
    for _ in range(3):
        fun2.zero_()
        nit2.zero_()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(nit2.cpu().numpy(), nit.cpu().numpy())
        np.testing.assert_allclose(fun2.cpu().numpy(), fun.cpu().numpy(),
                                   rtol=1e-11)


@pytest.mark.parametrize('evg', ['robust', 'classic'])
@pytest.mark.parametrize('n', [2, 24, 91, 92, 181, 182])
def test_bins_few_pairs(gpu, n, evg):
    """Steps whose passes run in one workgroup (up to 4 chunks of 4 096
    pairs: 181 stations) and beyond, with missing values and a step without
    any, against the oracle."""
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0, 2e5, n), rng.uniform(0, 2e5, n)
    vals = rng.gamma(2.0, 3.0, (3, n))
    vals[1, rng.choice(n, n // 3, replace=False)] = np.nan
    vals[2] = np.nan
    f = BatchVariogramFitter(x, y)
    bh, bg, bn, nb = (a.cpu().numpy() for a in f.empirical(vals, 0.5, 50, evg))
    assert nb[2] == 0
    for t in (0, 1):
        ok = ~np.isnan(vals[t])
        if ok.sum() < 2:
            continue
        ref = V.empirical(x[ok], y[ok], vals[t][ok], 0.5, 50, evg)
        k = nb[t]
        assert k == len(ref)
        np.testing.assert_array_equal(bn[t, :k], ref[:, 2])
        np.testing.assert_allclose(bh[t, :k], ref[:, 0], rtol=1e-12)
        np.testing.assert_allclose(bg[t, :k], ref[:, 1], rtol=1e-12)


def test_few_bins_and_many_give_the_same_bits(gpu):
    """Few bins evolve in one workgroup per candidate, many over the whole
    device: whichever takes a step, the result is the same to the last bit
    (here the whole device is chosen for the call by a step with many bins,
    the workgroup for the small steps alone and while capturing), and a fit of
    one bin, which never converges, takes no launch per generation."""
    import time
    import torch
    from spinterps_amd.variograms.fitvgs import BatchVariogramFitter
    rng = np.random.default_rng(5)
    n = 150
    x, y = rng.uniform(0, 2e5, n), rng.uniform(0, 2e5, n)
    vals = rng.gamma(2.0, 3.0, (4, n))
    for t, k in ((0, 9), (1, 14), (2, 25)):
        vals[t, k:] = np.nan
    f = BatchVariogramFitter(x, y)
    kw = dict(mdr=0.5, nk=20, perm_r_list=[1, 2], fit_vgs=['all'],
              fil_nug_vg='Nug', range_ub=2e5, opt_iters=40, seed=3,
              min_vld_stns=2, return_details=True)
    for t, lo, hi in ((0, 1, 3), (1, 2, 5), (2, 8, 12)):
        _, det = f.fit(vals[[t, 3]], **kw)
        _, one = f.fit(vals[[t]], **kw)
        nb = det['bins'][3].cpu().numpy()
        assert lo <= nb[0] <= hi and nb[1] > 100, nb
        # (the random streams are keyed on the step's place in the call)
        for k in ('params', 'fun', 'nit'):
            np.testing.assert_array_equal(one[k][0], det[k][0])
    kw.update(opt_iters=10000, nk=50, fit_vgs=['Sph', 'Exp', 'Gau'])
    f.fit(vals[:1], **kw)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    _, det = f.fit(vals[:1], **kw)
    # 1.2 ms; 200 ms with launches for each of up to 10 000 generations
    assert time.perf_counter() - t0 < 0.05, det['nit']
