"""The team placement against the oracle, bit for bit: row counts that do and
do not fill the wavefronts' slots, ensembles that do and do not fill a
workgroup, wide parameter rows, weights, claim orders and the resumed pilot."""

import numpy as np
import pytest

from menodax_amd import _kernels as K, rodas5P, tsit5
from menodax_amd._sparsity import normalize_sparsity
from oracle import oracle as O
from tests import systems as S
from tests.test_gpu_parity import _same, _structure

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_traj", [1, 64, 65, 200])
@pytest.mark.parametrize("n_osc", [9, 12, 32])
@pytest.mark.parametrize("kw", [{}, dict(refill=True), dict(work_order="pilot")],
                         ids=["plain", "refill", "pilot"])
def test_tsit5_ring(n_osc, n_traj, kw):
    n = 2 * n_osc
    fn, _ = S.vdp_lattice(n_osc, mu=1.0)
    assert K.tsit5_team(None, n, 1, fn)
    y0, p = S.vdp_scenario(n_osc, n_traj, 42, divergence=0.5)
    run = dict(first_step=1e-4, rtol=1e-6, atol=1e-8)
    hist, st = tsit5.solve(fn, y0, S.VDP_TIMES, p, return_stats=True, **run, **kw)
    _same(hist, st, *O.tsit5(O.vdp_lattice(n_osc, mu=1.0), y0, S.VDP_TIMES, p, **run))


@pytest.mark.parametrize("n", [17, 24, 50])
def test_tsit5_wide_parameters_weights_and_a_step_budget(n):
    fn, _, (rows, cols, vals, pidx) = S.arrow_system(n)
    system = O.linquad(n, rows, cols, vals, 0.01, pidx, S.arrow_n_params(n))
    y0, p = S.arrow_ensemble(70, n=n, lam_range=(1e-1, 1e2), rate_range=(0.05, 2.0))
    assert K.tsit5_team(None, n, p.shape[1], fn) and p.shape[1] > K.TEAM_PARAM_REGS
    t = np.linspace(0.0, 0.05, 5)
    w = np.random.default_rng(0).uniform(0.5, 2.0, size=(70, n))
    for max_steps in (100000, 6):
        run = dict(rtol=1e-6, atol=1e-8, max_steps=max_steps)
        hist, st = tsit5.solve(fn, y0, t, p, error_weights=w, return_stats=True, **run)
        ref, rst = O.tsit5(system, y0, t, p, weights=w, **run)
        reached = ~np.isnan(hist)
        assert reached.all() == (max_steps > 6)
        np.testing.assert_array_equal(hist[reached], ref[reached])
        for k in rst:
            np.testing.assert_array_equal(st[k], rst[k])


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("n_osc, n_traj", [(9, 1), (9, 65), (12, 64), (32, 100)])
@pytest.mark.parametrize("kw", [{}, dict(refill=True), dict(work_order="pilot")],
                         ids=["plain", "refill", "pilot"])
def test_rodas5p_ring(n_osc, n_traj, lu, kw):
    n, mask = 2 * n_osc, S.vdp_sparsity(n_osc)
    fn, _ = S.vdp_lattice(n_osc)
    assert K.rodas5p_team(fn, n, 1, K.KernelOptions(sparsity=normalize_sparsity(mask, n),
                                                    lu_precision=lu))
    y0, p = S.vdp_scenario(n_osc, n_traj, 42, divergence=0.25)
    run = dict(first_step=1e-4, rtol=1e-6, atol=1e-8, lu_precision=lu)
    hist, st = rodas5P.solve(fn, y0, S.VDP_TIMES, p, sparsity=mask, return_stats=True, **run, **kw)
    _same(hist, st, *O.rodas5p(O.vdp_lattice(n_osc), y0, S.VDP_TIMES, p,
                               layout=_structure(mask, n, "amd"), **run))


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [17, 24, 50])
def test_rodas5p_arrow_weights_budget_and_order(n, lu):
    fn, mask, (rows, cols, vals, pidx) = S.arrow_system(n)
    system = O.linquad(n, rows, cols, vals, 0.01, pidx, S.arrow_n_params(n))
    y0, p = S.arrow_ensemble(130, n=n, rate_range=(0.05, 5.0))
    t = np.linspace(0.0, 10.0, 6)
    w = np.random.default_rng(0).uniform(0.5, 2.0, size=(130, n))
    layout = _structure(mask, n, "amd")
    order = np.random.default_rng(1).permutation(130)
    for weights, max_steps, extra in ((None, 100000, {}), (w, 100000, dict(work_order=order)),
                                      (None, 30, dict(work_order="pilot")), (w, 30, {})):
        run = dict(rtol=1e-6, atol=1e-8, lu_precision=lu, max_steps=max_steps)
        hist, st = rodas5P.solve(fn, y0, t, p, sparsity=mask, error_weights=weights,
                                 return_stats=True, **run, **extra)
        _same(hist, st, *O.rodas5p(system, y0, t, p, weights=weights, layout=layout, **run))


def test_rodas5p_end_time_from_a_parameter():
    """The team reads the end-time column itself: the same bits as one lane a
    trajectory."""
    ring, mask = S.vdp_lattice(12)[0], S.vdp_sparsity(12)
    y0, p = S.vdp_scenario(12, 40, 42, divergence=0.25)
    p = np.column_stack([p, np.linspace(0.2, 1.0, 40)])
    run = dict(sparsity=mask, tf_index=1, rtol=1e-6, atol=1e-8, return_stats=True)
    hist, st = rodas5P.solve(ring, y0, S.VDP_TIMES, p, **run)
    ref, rst = rodas5P.solve(ring, y0, S.VDP_TIMES, p, placement="rolled", **run)
    _same(hist, st, ref, rst)


@pytest.mark.parametrize("n_traj", [64 * 256 + 1, 128 * 256 + 77])
def test_unrolled_workgroups_of_two_and_four_wavefronts(n_traj):
    y0, p = S.robertson_lognormal_ensemble(n_traj, seed=2)
    t = S.robertson_benchmark_times()[::7]
    run = dict(rtol=1e-6, atol=1e-8, return_stats=True)
    hist, st = rodas5P.solve(S.robertson, y0, t, p, **run)
    _same(hist, st, *O.rodas5p(O.robertson(), y0, t, p, rtol=1e-6, atol=1e-8))
