"""Tile autotuner of the batched and plain contractions: every variant of a
kernel family writes bit-identical results, so the tuned choice changes
only the time; the context reports what it timed and picked."""
import numpy as np
import pytest

from spinterps_amd import configs

pytestmark = pytest.mark.gpu


def _run(prob, vals, vgs, precision):
    import torch
    from spinterps_amd.interp.steps import interp_steps
    e, v, info = interp_steps(prob, vals, vgs, 'OK', precision=precision)
    torch.cuda.synchronize()
    return e.cpu().numpy(), v.cpu().numpy(), info.cpu().numpy()


def _same(outs):
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('family,precision,variants', [
    ('gemm_plain_f64', 'fp64', (0, 1, 2)),
    ('gemm_tri_bf16', 'mixed', (0, 1)),
])
def test_variants_bit_identical(gpu, family, precision, variants):
    """Each forced variant (k depth 8 / 16 / 32 of the plain FP64
    contraction; delta loaded after or during the products of the
    split-BF16 contraction) gives the same estimates, variances and flags
    on hourly steps of 200-2 000 stations."""
    from spinterps_amd._lib import context
    from spinterps_amd.interp.steps import DeviceProblem
    w = configs.hourly(n_side=128, cell=500.0)
    T = 6 if precision == 'fp64' else 32
    vals, vgs = configs.hourly_steps(w, 0, T)
    prob = DeviceProblem.from_workload(w)
    ctx = context(0)
    outs = []
    try:
        for v in variants:
            ctx.force_variant(family, v)
            outs.append(_run(prob, vals, vgs, precision))
    finally:
        ctx.force_variant(family, -1)
    _same(outs)


def test_autotune_picks_and_reports(gpu):
    """With tuning on, the first launches of each size class time every
    variant and keep the fastest; results equal the untuned defaults, and
    a class is timed once per context."""
    from spinterps_amd import _lib
    from spinterps_amd.interp.steps import DeviceProblem
    w = configs.hourly(n_side=128, cell=500.0)
    vals, vgs = configs.hourly_steps(w, 100, 132)
    prob = DeviceProblem.from_workload(w)
    ctx = _lib.context(0)
    ctx.set_tuning(False)
    try:
        ref_m = _run(prob, vals, vgs, 'mixed')
        ref_p = _run(prob, vals[:4], vgs[:4], 'fp64')
        before = ctx.tuning_report()
        ctx.set_tuning(True)
        got_m = _run(prob, vals, vgs, 'mixed')
        got_p = _run(prob, vals[:4], vgs[:4], 'fp64')
        rep = ctx.tuning_report()
        _same([ref_m, got_m])
        _same([ref_p, got_p])
        fams = {'gemm_plain_f64': 3, 'gemm_tri_bf16': 2}
        assert {r[0] for r in rep} == set(fams), rep
        for fam, cls, choice, ms in rep:
            assert len(ms) == fams[fam] and 0 <= choice < fams[fam], rep
            assert cls >= 1 and all(t > 0 for t in ms), rep
            assert ms[choice] == min(ms), rep
        keys = [(r[0], r[1]) for r in rep]
        assert len(keys) == len(set(keys)), rep
        assert len(rep) >= len(before)
        # a second call times nothing new
        _run(prob, vals, vgs, 'mixed')
        assert ctx.tuning_report() == rep
        print('tuned:', rep)
    finally:
        ctx.set_tuning(True)


def test_tuning_arguments_checked(gpu):
    from spinterps_amd import _lib
    ctx = _lib.context(0)
    with pytest.raises(AssertionError):
        ctx.force_variant('gemm_nothing', 0)
    with pytest.raises(AssertionError):
        ctx.force_variant('gemm_plain_f64', 3)
    with pytest.raises(AssertionError):
        _lib.check(_lib.lib().spk_ctx_set_tuning(ctx.h, 7))


def test_tuning_times_a_step_with_a_system(gpu):
    """Of the steps with the most stations the one that is timed has a
    system: with the last of them below the threshold (mean-filled, no
    kernel runs), the times are those of the same call without it."""
    from spinterps_amd import _lib
    from spinterps_amd.interp.steps import DeviceProblem
    rng = np.random.default_rng(2)
    n = 1000
    g = np.linspace(0, 1e5, 300)
    gx, gy = np.meshgrid(g, g)
    prob = DeviceProblem(*rng.uniform(0, 1e5, (2, n)), gx.ravel(), gy.ravel())
    vals = rng.gamma(2.0, 5.0, (2, n))
    vgs = ['0.5 Nug(0.0) + 9.0 Exp(30000.0)'] * 2
    fill = vals.copy()
    fill[1] *= 1e-3
    own, ms = _lib._ctxs.get(0), []
    try:
        for v in (vals, fill):
            _lib._ctxs[0] = _lib.Context(0)
            from spinterps_amd.interp.steps import interp_steps
            interp_steps(prob, v, vgs, 'OK', min_var_thr=1.0)
            ms.append([r[3] for r in _lib._ctxs[0].tuning_report()
                       if r[0] == 'gemm_plain_f64'])
    finally:
        _lib._ctxs[0] = own
        if own is None:
            del _lib._ctxs[0]
    # 1.5 ms and more each; empty launches take a few microseconds
    assert min(ms[1][0]) > 0.5 * min(ms[0][0]), ms
