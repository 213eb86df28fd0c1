"""Neighbourhood interpolation (nrst / pie, interp/grps.py:141-288,
interp/steps.py:592-608, 732-831) on the GPU against oracle.interp_all
(GPU)."""
import numpy as np
import pytest

from oracle import spk_oracle as O
from spinterps_amd import _lib

pytestmark = pytest.mark.gpu

OX, OY = 350000.0, 5300000.0


def _case(seed=7, n=120, side=24, T=8, dup=False):
    """n stations on 100 km x 100 km plus two far ones (never selected:
    dropped), side x side cells, T steps: missing stations, one step with a
    single station, one without any, low values in the west so that some
    neighbourhoods are mean-filled; optionally two stations at one place
    (singular covariance blocks: the pseudo-inverse fallback)."""
    rng = np.random.default_rng(seed)
    sx = np.r_[OX + rng.uniform(0, 1e5, n), OX + 9e5, OX - 6e5]
    sy = np.r_[OY + rng.uniform(0, 1e5, n), OY + 8e5, OY - 7e5]
    if dup:
        sx[1], sy[1] = sx[0], sy[0]
    N = sx.size
    cell = 1e5 / side
    g = np.arange(side) * cell + cell / 2
    cx, cy = [a.ravel() for a in np.meshgrid(OX + g, OY + g[::-1])]
    z = rng.gamma(0.8, 5.0, (T, N)) + 0.05
    west = sx < OX + 3e4
    z[:, west] = rng.uniform(0.0, 0.3, (T, int(west.sum())))
    z[1, rng.choice(n, n // 5, replace=False)] = np.nan
    z[2, :] = np.nan
    z[2, 17] = 3.5                      # one station
    z[3, :] = np.nan                    # none
    z[5, rng.choice(n, 40, replace=False)] = np.nan
    models = ['Sph', 'Exp', 'Gau', 'Sph', 'Exp', 'Gau', 'Sph', 'Exp']
    vgs = []
    for t in range(T):
        v = float(np.nanvar(z[t])) if np.isfinite(z[t]).sum() > 1 else 1.0
        vgs.append(f'{0.1 * v!r} Nug(0.0) + {0.9 * v!r} '
                   f'{models[t]}({float(rng.uniform(2e4, 6e4))!r})')
    drift = np.sin(sx / 2e4) * 300.0 + sy / 1e3 - OY / 1e3
    cdrift = np.sin(cx / 2e4) * 300.0 + cy / 1e3 - OY / 1e3
    return sx, sy, cx, cy, z, vgs, drift, cdrift


def _run(gpu, case, method, sel, n_nebs, n_pies=None, thr=0.5):
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    sx, sy, cx, cy, z, vgs, drift, cdrift = case
    edk = method == 'EDK'
    prob = DeviceProblem(sx, sy, cx, cy,
                         stn_drift=drift[:, None] if edk else None,
                         cell_drift=cdrift[None, :] if edk else None)
    e, v, info = interp_neb_steps(prob, z, vgs, method, neb_sel_mthd=sel,
                                  n_nebs=n_nebs, n_pies=n_pies,
                                  min_var_thr=thr)
    _, f64, prb = O.interp_all(
        sx, sy, cx, cy, z, vgs, [(method, method, 2.0)],
        stn_drfts=drift[:, None] if edk else None,
        cell_drfts=cdrift[None, :] if edk else None, min_var_thr=thr,
        neb_sel_mthd=sel, n_nebs=n_nebs, n_pies=n_pies)
    return (e.cpu().numpy(), None if v is None else v.cpu().numpy(),
            info.cpu().numpy(), f64, prb)


def _close(got, ref, scale, rtol, what):
    assert np.array_equal(np.isnan(got), np.isnan(ref)), what
    ok = ~np.isnan(ref)
    err = np.abs(got[ok] - ref[ok]).max() / scale
    assert err <= rtol, (what, err)


@pytest.mark.parametrize('sel,n_nebs,n_pies', [('nrst', 10, None),
                                                ('nrst', 50, None),
                                                ('pie', 12, 4)])
def test_ok_matches_oracle(gpu, sel, n_nebs, n_pies):
    case = _case()
    e, v, info, f64, prb = _run(gpu, case, 'OK', sel, n_nebs, n_pies)
    z = case[4]
    scale = np.nanmax(np.abs(z))
    # FP64 Cholesky against the oracle's pinv on well-conditioned sets
    _close(e, f64['OK'], scale, 1e-9, 'est')
    _close(v, f64['EST_VARS_OK'], np.nanmax(f64['EST_VARS_OK']), 1e-8, 'var')
    assert sorted(prb) == [3]
    assert info[3] == _lib.ST_NOSTNS
    if sel == 'nrst':
        assert info[2] & _lib.ST_ONESTN    # one station: copied, var NaN
        assert np.all(e[2] == 3.5) and np.all(np.isnan(v[2]))
    else:
        # pie repeats the one station n_nebs times (numpy's broadcast in
        # interp/grps.py:245): a singular set, solved by the pseudo-inverse
        assert info[2] & _lib.ST_PINV
        np.testing.assert_allclose(e[2], 3.5, rtol=1e-12)
    # mean-filled groups (variance 0) flagged where the oracle has them
    fill = [bool((f64['EST_VARS_OK'][t] == 0.0).any()) for t in (0, 1, 4)]
    assert [bool(info[t] & 2) for t in (0, 1, 4)] == fill
    if n_nebs == 10:
        assert any(fill)
    assert not any(info[t] & (4 | 16 | 128) for t in range(len(info))
                   if t != 2)


@pytest.mark.parametrize('method', ['IDW', 'NNB', 'SK', 'SKM', 'EDK'])
def test_other_methods_match_oracle(gpu, method):
    case = _case(seed=3)
    e, v, info, f64, prb = _run(gpu, case, method, 'nrst', 12)
    scale = np.nanmax(np.abs(case[4]))
    # EDK's bordered system holds drifts of a few hundred against
    # covariances of about ten: the oracle's pinv carries ~1e-9 there
    tol = {'NNB': 0.0, 'EDK': 1e-8}.get(method, 1e-9)
    _close(e, f64[method], scale, tol, method)
    assert v is None


@pytest.mark.parametrize('method', ['OK', 'SK', 'EDK'])
@pytest.mark.parametrize('n_nebs', [2, 13, 14, 15, 16, 29, 30, 31, 45, 46, 47,
                                    48, 54, 55, 58, 60])
def test_set_sizes_match_oracle(gpu, method, n_nebs):
    """Set sizes around the 16-row blocks of the chunk kernel and its limit,
    with one-model, two-model, linear and unbounded variograms.  The
    covariance matrices' condition numbers stay below 1e4 (the Gaussian
    model's with a range of 12 km near the station spacing; 3e7 at 50 km), so
    k 2^-53 cond is below 1e-10; EDK's border adds a factor."""
    case = list(_case(n=90, side=6, T=8, seed=n_nebs))
    v = [float(x.split()[0]) * 10.0 for x in case[5]]
    case[5][4] = f'{0.6 * v[4]!r} Sph(2e4) + {0.4 * v[4]!r} Exp(7e4)'
    case[5][5] = f'{0.1 * v[5]!r} Nug(0.0) + {0.9 * v[5]!r} Gau(1.2e4)'
    if method != 'EDK':
        # (with a drift the linear model, not positive definite in the plane,
        # gives bordered matrices with condition numbers of 3e6 and more)
        case[5][6] = f'{0.2 * v[6]!r} Nug(0.0) + {0.8 * v[6]!r} Lin(5e4)'
    if method == 'OK':
        # (for EDK in metres the condition number is 2e11)
        case[5][7] = f'{v[7]!r} Rng(1.0)'
    if method == 'EDK' and n_nebs < 4:
        pytest.skip('two stations do not determine mean and drift')
    e, var, info, f64, prb = _run(gpu, case, method, 'nrst', n_nebs, thr=0.0)
    scale = np.nanmax(np.abs(case[4]))
    _close(e, f64[method], scale, {'EDK': 1e-8}.get(method, 1e-9), method)
    if method == 'OK':
        _close(var, f64['EST_VARS_OK'], np.nanmax(f64['EST_VARS_OK']), 1e-8,
               'var')
    # solved by the sweep itself, not by the pseudo-inverse that takes the
    # chunks it rejects (and that agrees with the oracle anyway); the linear
    # model is not positive definite in the plane, some of its sets fail
    for t in (0, 1, 4, 5) + ((6,) if method == 'EDK' else ()):
        assert not info[t] & (_lib.ST_PINV | _lib.ST_ILLCOND), (t, info[t])


@pytest.mark.parametrize('method,drifts', [('OK', 0), ('SK', 0), ('SKM', 0),
                                           ('EDK', 1), ('EDK', 2),
                                           ('EDK', 3), ('EDK', 7)])
@pytest.mark.parametrize('n_nebs', [40, 47, 54, 58])
def test_chunks_of_many_cells(gpu, method, drifts, n_nebs):
    """One set for all cells: chunks of 64, 64 and 41 cells, which take one
    chunk kernel or the other by their groups of cells (one-model and
    two-model variograms in calls of their own), against the exact solution
    of the same systems.  Covariance matrices of condition 1e4 and less, the
    drifts of order one: k 2^-53 cond is below 1e-10, 1e-9 with the border."""
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    rng = np.random.default_rng(n_nebs)
    n = n_nebs
    sx, sy = rng.uniform(0, 1e5, n), rng.uniform(0, 1e5, n)
    g = np.arange(13) * 8e3 + 1e3
    cx, cy = [a.ravel() for a in np.meshgrid(g, g)]
    m = drifts

    def drift(x, y):
        return np.stack([np.sin((x + k * y) / (2e4 + 5e3 * k))
                         for k in range(m)])
    z = rng.gamma(2.0, 5.0, (2, n))
    for vgs in (['0.5 Nug(0.0) + 9.0 Exp(30000.0)', '9.0 Sph(40000.0)'],
                ['4.0 Sph(20000.0) + 5.0 Exp(60000.0)', '9.0 Sph(40000.0)']):
        sd, cd = (drift(sx, sy).T.copy(), drift(cx, cy)) if m else (None, None)
        prob = DeviceProblem(sx, sy, cx, cy, sd, cd)
        e, v, info = interp_neb_steps(prob, z, vgs, method,
                                      neb_sel_mthd='nrst', n_nebs=n)
        for t in range(2):
            assert not int(info[t]) & (_lib.ST_PINV | _lib.ST_ILLCOND)
            dd = O.dists_2d(sx, sy, sx, sy)
            rd = O.dists_2d(cx, cy, sx, sy)
            if method == 'SK':
                K, R = O.krig_system('SK', vgs[t], dd, rd, None, None, 0.0)
                ref, var = O.krige_solve(K, R, z[t], rd, False)[:2]
            else:
                ref, var, _ = O.krige_exact(method, vgs[t], dd, rd, z[t], sd,
                                            cd, want_var=method == 'OK')
            _close(e[t].cpu().numpy(), ref, np.abs(z).max(), 1e-9, method)
            if method == 'OK':
                _close(v[t].cpu().numpy(), var, var.max(), 1e-9, 'var')


def test_variance_rounding(gpu):
    """The variance c0 - |y|^2 + ... of sets of 50 against long double: with
    |y|^2 summed by eights its error is 4.7e-16 of the variances' size (term by
    term, the rounding growing over all 50, 5.2e-16)."""
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    LD = np.longdouble
    rng = np.random.default_rng(12)
    n, K, C, q = 400, 50, 240, 2.0 ** 20
    sx, sy = np.round(rng.uniform(0, 4e5, (2, n)) * q) / q
    cx, cy = np.round(rng.uniform(0, 4e5, (2, C)) * q) / q
    z = rng.gamma(2.0, 5.0, (1, n))
    vg = '1.5 Sph(50000.0) + 8.5 Exp(75000.0)'
    _, v, info = interp_neb_steps(DeviceProblem(sx, sy, cx, cy), z, [vg],
                                  'OK', neb_sel_mthd='nrst', n_nebs=K)
    assert not int(info[0]) & (_lib.ST_PINV | _lib.ST_ILLCOND)

    def gam(h):
        h = LD(h)
        a = h / LD(50000)
        sph = np.where(a >= 1, LD(1), LD(1.5) * a - a ** 3 / 2)
        return LD(1.5) * sph - LD(8.5) * np.expm1(-3 * h / LD(75000))

    def dist(x0, y0, x1, y1):
        return np.sqrt((LD(x0)[:, None] - LD(x1)) ** 2
                       + (LD(y0)[:, None] - LD(y1)) ** 2)
    ref = np.zeros(C, LD)
    d = np.hypot(cx[:, None] - sx, cy[:, None] - sy)
    for c in range(C):
        s = np.sort(np.argsort(d[c], kind='stable')[:K])
        A = np.ones((K + 1, K + 1), LD)
        A[K, K] = 0
        A[:K, :K] = gam(dist(sx[s], sy[s], sx[s], sy[s]))
        r = np.ones(K + 1, LD)
        r[:K] = gam(dist(cx[c:c + 1], cy[c:c + 1], sx[s], sy[s])[0])
        Ad = np.linalg.inv(A.astype(float))
        x = LD(Ad @ r.astype(float))
        for _ in range(4):
            x = x + LD(Ad @ (r - A @ x).astype(float))
        ref[c] = x[:K] @ r[:K] + 2 * x[K]
    err = LD(v[0].cpu().numpy()) - ref
    rel = float(np.sqrt((err ** 2).sum() / (ref ** 2).sum()))
    assert rel < 5.0e-16, rel


@pytest.mark.parametrize('k', [1, 3, 8])
def test_tiles_of_exactly_k_candidates(gpu, k):
    """Tiles of cells that no more than k stations can reach: all are taken
    (clusters of k stations far apart, the cells of a cluster around it)."""
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    rng = np.random.default_rng(k)
    ox, oy = np.meshgrid(np.arange(4) * 1e6, np.arange(4) * 1e6)
    sx = (ox.ravel()[:, None] + rng.uniform(0, 1e3, (16, k))).ravel()
    sy = (oy.ravel()[:, None] + rng.uniform(0, 1e3, (16, k))).ravel()
    cx = (ox.ravel()[:, None] + rng.uniform(0, 1e3, (16, 64))).ravel()
    cy = (oy.ravel()[:, None] + rng.uniform(0, 1e3, (16, 64))).ravel()
    z = rng.gamma(2.0, 5.0, (1, sx.size))
    e, _, _ = interp_neb_steps(DeviceProblem(sx, sy, cx, cy), z, None, 'IDW',
                               neb_sel_mthd='nrst', n_nebs=k)
    d = np.hypot(cx[:, None] - sx, cy[:, None] - sy)
    at = np.argsort(d, axis=1)[:, :k]
    w = 1.0 / np.take_along_axis(d, at, 1) ** 2
    ref = (w * z[0][at]).sum(1) / w.sum(1)
    np.testing.assert_allclose(e[0].cpu().numpy(), ref, rtol=1e-12)


@pytest.mark.parametrize('n,k', [(71, 30), (51, 50), (65, 64), (701, 20)])
def test_cells_without_finite_distances(gpu, n, k):
    """Cells at infinity, beyond 1e154 or without a coordinate beside others in
    a tile: their sets are the first k active stations, the others' results
    are as without them (some of many candidates, all of exactly k, more sets
    than fit the sweep, more candidates than are staged)."""
    from spinterps_amd.interp.steps import (DeviceProblem, interp_neb_steps,
                                            interp_steps)
    rng = np.random.default_rng(n + k)
    sx, sy = rng.uniform(0, 1e5, n), rng.uniform(0, 1e5, n)
    cx, cy = rng.uniform(0, 1e5, 200), rng.uniform(0, 1e5, 200)
    z = rng.gamma(2.0, 3.0, (1, n))
    z[0, 2] = np.nan
    vg = ['0.1 Nug(0.0) + 2.0 Sph(60000.0)']
    fx, fy = cx.copy(), cy.copy()
    fx[9], fy[11], fy[70], fx[130] = 1.7e308, np.inf, 1e200, np.nan

    def run(x, y):
        e, v, _ = interp_neb_steps(DeviceProblem(sx, sy, x, y), z, vg, 'OK',
                                   neb_sel_mthd='nrst', n_nebs=k)
        return e.cpu().numpy()[0], v.cpu().numpy()[0]

    want, got = run(cx, cy), run(fx, fy)
    own = np.setdiff1d(np.arange(200), (9, 11, 70, 130))
    first = np.setdiff1d(np.arange(n), (2,))[:k]
    e, v, _ = interp_steps(
        DeviceProblem(sx[first], sy[first], np.array([1e9]), np.array([1e9])),
        z[:, first], vg, 'OK')
    for g, w, f in zip(got, want, (e.cpu().numpy(), v.cpu().numpy())):
        np.testing.assert_allclose(g[own], w[own], rtol=1e-11)
        np.testing.assert_allclose(g[[9, 11, 70]], f[0, 0], rtol=1e-11)


def test_edk_reproduces_the_drift(gpu):
    """Values that are a linear function of the drift are reproduced at
    every cell (the weights sum to one and reproduce the drift)."""
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    sx, sy, cx, cy, z, vgs, drift, cdrift = _case(seed=3)
    z = np.where(np.isnan(z), np.nan, 2.0 + 0.5 * drift[None, :])
    z[:, -2:] = np.nan           # the far stations
    prob = DeviceProblem(sx, sy, cx, cy, stn_drift=drift[:, None],
                         cell_drift=cdrift[None, :])
    e, _, info = interp_neb_steps(prob, z, vgs, 'EDK', neb_sel_mthd='nrst',
                                  n_nebs=12)
    e = e.cpu().numpy()
    for t in (0, 1, 4, 5, 6, 7):
        np.testing.assert_allclose(e[t], 2.0 + 0.5 * cdrift, rtol=1e-9,
                                   atol=1e-9 * np.abs(cdrift).max())


def test_every_station_equals_all_path(gpu):
    """n_nebs at least the active count: one neighbourhood per step, so the
    results are the 'all' path's (FP64 plain) within rounding."""
    from spinterps_amd.interp.steps import (DeviceProblem, interp_neb_steps,
                                            interp_steps)
    sx, sy, cx, cy, z, vgs, _, _ = _case(n=40)
    sx, sy, z = sx[:40], sy[:40], z[:, :40]
    prob = DeviceProblem(sx, sy, cx, cy)
    e1, v1, i1 = interp_neb_steps(prob, z, vgs, 'OK', neb_sel_mthd='nrst',
                                  n_nebs=64, min_var_thr=0.5)
    e2, v2, i2 = interp_steps(prob, z, vgs, 'OK', precision='fp64',
                              min_var_thr=0.5)
    e1, v1, e2, v2 = [a.cpu().numpy() for a in (e1, v1, e2, v2)]
    _close(e1, e2, np.nanmax(np.abs(z)), 1e-9, 'est')
    _close(v1, v2, np.nanmax(v2), 1e-8, 'var')


def test_singular_sets_use_the_pseudo_inverse(gpu):
    """Two stations at one place make every set holding both singular: the
    Cholesky fails and the group is solved by pinv of the bordered system,
    as the reference solves it."""
    case = _case(seed=5, dup=True)
    z = case[4]
    z[:, 1] = z[:, 0]            # one value per place, as a real duplicate
    e, v, info, f64, prb = _run(gpu, case, 'OK', 'nrst', 10)
    scale = np.nanmax(np.abs(z))
    # both sides drop the exact null vector of the duplicate; the kept
    # spectrum of such sets spans about 1e8, so the two pseudo-inverses
    # (an SVD here, a symmetric eigendecomposition there) agree to ~1e-8
    _close(e, f64['OK'], scale, 1e-7, 'est')
    _close(v, f64['EST_VARS_OK'], np.nanmax(f64['EST_VARS_OK']), 1e-7, 'var')
    # with a dropped eigenvalue the sets are flagged ill-conditioned
    assert info[0] & _lib.ST_PINV and info[0] & _lib.ST_ILLCOND


@pytest.mark.parametrize('n_nebs,n_pies', [(1, 1), (9, 1), (24, 3), (24, 24),
                                           (40, 33), (64, 64), (50, 2)])
def test_pie_sector_counts(gpu, n_nebs, n_pies):
    """Sector counts around the powers of two that split the wavefront; sets
    of the wrong stations would be off by far more than rounding."""
    case = list(_case(n=150, side=7))
    case[4][2] = case[4][0]
    e, _, info, f64, prb = _run(gpu, case, 'IDW', 'pie', n_nebs, n_pies,
                                thr=0.0)
    _close(e, f64['IDW'], np.nanmax(np.abs(case[4])), 1e-12, 'IDW')


def test_pie_with_too_few_stations_is_refused(gpu):
    from spinterps_amd.interp.steps import DeviceProblem, interp_neb_steps
    sx, sy, cx, cy, z, vgs, _, _ = _case()
    z = z.copy()
    z[0, 5:] = np.nan            # five active stations, twelve wanted
    prob = DeviceProblem(sx, sy, cx, cy)
    with pytest.raises(Exception, match='fewer active stations'):
        interp_neb_steps(prob, z[:1], vgs[:1], 'OK', neb_sel_mthd='pie',
                         n_nebs=12, n_pies=4)
