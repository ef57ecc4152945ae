"""The adjoint's stores, bit for bit: a record of every step in the LDS form of
the rolled adjoint, the plain record against the forms that need no checkpoints
(the stage-keeping kernel and the team's), and a trajectory that outruns such a
form's store."""

import numpy as np
import pytest

from menodax_amd import _autodiff, _kernels as K, rodas5P
from menodax_amd._sparsity import normalize_sparsity
from tests import systems as S

pytestmark = pytest.mark.gpu


def _launches(monkeypatch):
    """Notes each adjoint launch: its kernel's source, checkpoints, whether the
    store was enough."""
    runs = []
    real = _autodiff._adjoint_run

    def spy(job, *a, adjoint=None, **k):
        out = real(job, *a, adjoint=adjoint, **k)
        runs.append(((adjoint or job.adjoint()).source, a[3], out is not None))
        return out

    monkeypatch.setattr(_autodiff, "_adjoint_run", spy)
    return runs


def _lattice(n_osc, traj):
    fn, _ = S.vdp_lattice(n_osc, mu=1.0, d=0.1, wrap=False)
    y0, p = S.vdp_scenario(n_osc, traj, 3, divergence=0.9)
    return fn, y0, p, np.array([0.0, 0.5, 0.500001, 0.500002, 2.9, 3.0])


def _gradients(fn, y0, t, p, **kw):
    import torch

    dev = torch.device("cuda")
    y = torch.tensor(y0, device=dev, requires_grad=True)
    q = torch.tensor(p, device=dev, requires_grad=True)
    hist, st = rodas5P.solve(fn, y, t, q, adjoint=True, return_stats=True, **kw)
    g = torch.as_tensor(np.random.default_rng(0).normal(size=tuple(hist.shape)), device=dev)
    (hist * g).sum().backward()
    got = y.grad.cpu().numpy(), q.grad.cpu().numpy()
    assert np.isfinite(got[0]).all() and np.isfinite(got[1]).all()
    assert int(st["accepted_steps"].max()) > 64
    return got


def _same(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("system, traj", [("dense 10", 70), ("dense 16", 33), ("sparse 12", 70)])
def test_the_lds_adjoint_records_every_step(system, traj, lu, monkeypatch):
    kind, n = system.split()
    n = int(n)
    if kind == "dense":
        fn, y0, p, t = _lattice(n // 2, traj)
        kw = dict(rtol=1e-9, atol=1e-11)
    else:  # more parameters than the team's adjoint sums
        fn, mask, _ = S.arrow_system(n)
        y0, p = S.arrow_ensemble(traj, n=n, lam_range=(1e-1, 1e3))
        assert p.shape[1] > K.ADJOINT_TEAM_MAX_PARAMS
        t, kw = np.linspace(0.0, 2.0, 6), dict(rtol=1e-7, atol=1e-9, sparsity=mask)
    runs = _launches(monkeypatch)
    got = _gradients(fn, y0, t, p, lu_precision=lu, **kw)
    ref = _gradients(fn, y0, t, p, lu_precision=lu, placement="rolled", **kw)
    (source, ckpts, fit), (rolled, rolled_ckpts, _) = runs
    assert "#define MDX_ADJ_LDS 1" in source and "#define MDX_ADJ_RECORD 1" in source
    assert ckpts == 1 and fit
    assert "#define MDX_ADJ_RECORD 0" in rolled and rolled_ckpts > 1
    _same(got, ref)


@pytest.mark.parametrize("n_osc, mark", [(1, "#define MDX_ADJ_KEEP 1"), (10, "#define MDX_TEAM ")])
def test_the_plain_record_and_the_forms_without_checkpoints(n_osc, mark, monkeypatch):
    fn, y0, p, t = _lattice(n_osc, 70)
    kw = dict(rtol=1e-10, atol=1e-12, lu_precision="fp64",
              sparsity=S.vdp_sparsity(n_osc, wrap=False) if n_osc > 1 else None)
    runs = _launches(monkeypatch)
    whole = _gradients(fn, y0, t, p, **kw)
    monkeypatch.setattr(rodas5P, "_whole_adjoint", lambda *a: {})
    plain = _gradients(fn, y0, t, p, **kw)
    assert mark in runs[0][0] and mark not in runs[1][0]
    assert "#define MDX_ADJ_RECORD 1" in runs[1][0]
    assert [(ckpts, fit) for _, ckpts, fit in runs] == [(1, True), (1, True)]
    _same(plain, whole)


@pytest.mark.parametrize("n_osc, mark", [(1, "#define MDX_ADJ_KEEP 1"), (10, "#define MDX_TEAM ")])
def test_a_store_that_is_outrun(n_osc, mark, monkeypatch):
    """Too few records for the longest trajectories: the launch reports it and
    the checkpoints give the same gradients."""
    fn, y0, p, t = _lattice(n_osc, 70)
    n = 2 * n_osc
    kw = dict(rtol=1e-10, atol=1e-12, lu_precision="fp64",
              sparsity=S.vdp_sparsity(n_osc, wrap=False) if n_osc > 1 else None)
    g = np.random.default_rng(1).normal(size=(70, t.size, n))
    _, st = rodas5P.solve(fn, y0, t, p, return_stats=True, **kw)
    steps = np.sort(st["accepted_steps"])
    room = int(steps[35])
    assert steps[0] < room < steps[-1]
    runs = _launches(monkeypatch)
    ref = rodas5P.adjoint_gradients(fn, y0, t, p, g, **kw)
    monkeypatch.setattr(_autodiff, "_record_store_guess",
                        lambda job: -(-room * job.whole_words // (job.n_vars + 4)))
    got = rodas5P.adjoint_gradients(fn, y0, t, p, g, **kw)
    assert [fit for _, _, fit in runs] == [True, False, True]
    assert mark in runs[0][0] and mark in runs[1][0] and mark not in runs[2][0]
    assert np.isfinite(ref[0]).all() and np.isfinite(ref[1]).all()
    _same(got, ref)
