"""The adjoint shared out over a workgroup's wavefronts against the rolled
scratch kernel, bit for bit: row counts that do and do not fill the slots, both
workgroup sizes, ensembles that do and do not fill a workgroup, trajectories of
very different step counts, rejected steps, saves within and past a step, error
weights, a step budget, several parameters and an end time from one of them."""

import numpy as np
import pytest

from menodax_amd import _kernels as K, rodas5P
from menodax_amd._sparsity import normalize_sparsity
from tests import systems as S

pytestmark = pytest.mark.gpu


def lattice(n_osc):
    """A chain of oscillators whose stiffness, coupling and decay are p[0..2];
    p[3] is not read by it."""
    terms = []
    for o in range(n_osc):
        x, v = 2 * o, 2 * o + 1
        couple = " + ".join([f"p[1] * (y[{2 * q}] - y[{x}])" for q in (o - 1, o + 1)
                             if 0 <= q < n_osc])
        terms += [f"y[{v}]", f"p[0] * (1.0 - y[{x}] * y[{x}]) * y[{v}] - y[{x}] + {couple}"
                             f" - p[2] * y[{v}] / (1.0 + y[{x}] * y[{x}])"]
    return S.make_tuple_callback("lattice", terms)


@pytest.mark.parametrize("n_osc, traj, block, lu, weighted", [
    (5, 1, 32, "fp64", False), (7, 33, 32, "fp32", True), (10, 96, 32, "fp64", True),
    (16, 70, 32, "fp32", False), (24, 17, 16, "fp64", False)])
def test_the_same_gradients(n_osc, traj, block, lu, weighted):
    import torch

    n = 2 * n_osc
    fn, mask = lattice(n_osc), S.vdp_sparsity(n_osc, wrap=False)
    options = K.KernelOptions(lu_precision=lu, sparsity=normalize_sparsity(mask, n), tf_index=3)
    assert K.rodas5p_adjoint_team(fn, n, 4, options, traj, 256) == block
    rng = np.random.default_rng(n)
    y0 = rng.uniform(-2.0, 2.0, (traj, n))
    p = np.column_stack([10.0 ** rng.uniform(-1.0, 1.5, traj), rng.uniform(0.05, 0.2, traj),
                         rng.uniform(0.0, 0.3, traj), rng.uniform(0.3, 1.0, traj)])
    t = np.array([0.0, 0.01, 0.011, 0.4, 0.9, 1.0])
    dev = torch.device("cuda")
    g = torch.as_tensor(rng.normal(size=(traj, 6, n)), device=dev)
    w = rng.uniform(0.5, 2.0, (traj, n)) if weighted else None

    def gradients(**kw):
        y = torch.tensor(y0, device=dev, requires_grad=True)
        q = torch.tensor(p, device=dev, requires_grad=True)
        hist, st = rodas5P.solve(fn, y, t, q, adjoint=True, return_stats=True, lu_precision=lu,
                                 sparsity=mask, tf_index=3, **kw)
        reached = ~torch.isnan(hist)
        (hist[reached] * g[reached]).sum().backward()
        return y.grad.cpu().numpy(), q.grad.cpu().numpy(), st

    for kw in (dict(rtol=1e-6, atol=1e-8, first_step=0.3), dict(rtol=1e-8, atol=1e-10, error_weights=w),
               dict(rtol=1e-6, atol=1e-8, max_steps=12)):
        got, ref = gradients(**kw), gradients(placement="rolled", **kw)
        if "first_step" in kw:
            assert (ref[2]["rejected_steps"] > 0).any()
        assert np.isfinite(ref[0]).all() and np.isfinite(ref[1]).all() and (ref[1][:, :3] != 0).all()
        np.testing.assert_array_equal(got[0], ref[0])
        np.testing.assert_array_equal(got[1], ref[1])
