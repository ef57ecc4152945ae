"""The adjoint that records every step in its forward pass against the one that
replays segments from checkpoints, bit for bit: the register step, the rolled
step in LDS and Tsit5, with trajectories of very different step counts and an
ensemble that leaves the last workgroup partly empty."""

import numpy as np
import pytest

from menodax_amd import _autodiff, rodas5P, tsit5
from tests import systems as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver, n_osc", [(rodas5P, 1), (rodas5P, 3), (rodas5P, 10), (tsit5, 1)],
                         ids=["rodas5P registers", "rodas5P 6 variables", "rodas5P team", "tsit5"])
def test_the_same_gradients(solver, n_osc, monkeypatch):
    import torch

    n, traj = 2 * n_osc, 70
    fn, _ = S.vdp_lattice(n_osc, mu=1.0, d=0.1, wrap=False)
    y0, mu = S.vdp_scenario(n_osc, traj, 3, divergence=0.9)
    dev = torch.device("cuda")
    t = np.array([0.0, 0.5, 0.500001, 0.500002, 2.9, 3.0])  # several saves in a step
    kw = dict(rtol=1e-10, atol=1e-12)
    if solver is rodas5P:
        kw.update(lu_precision="fp64",
                  sparsity=S.vdp_sparsity(n_osc, wrap=False) if n_osc > 1 else None)
    g = torch.as_tensor(np.random.default_rng(0).normal(size=(traj, 6, n)), device=dev)
    runs = []
    real = _autodiff._adjoint_run

    def spy(job, *a, **k):
        runs.append((a[3], k.get("ckpt_every")))
        return real(job, *a, **k)

    monkeypatch.setattr(_autodiff, "_adjoint_run", spy)

    def gradients(ckpt_every):
        y = torch.tensor(y0, device=dev, requires_grad=True)
        p = torch.tensor(mu, device=dev, requires_grad=True)
        hist, st = solver.solve(fn, y, t, p, adjoint=True, ckpt_every=ckpt_every,
                                return_stats=True, **kw)
        (hist * g).sum().backward()
        return y.grad.cpu().numpy(), p.grad.cpu().numpy(), int(st["accepted_steps"].max())

    whole = gradients(64)
    assert whole[2] > 64 and [r[0] for r in runs] == [1] and runs[0][1] > whole[2]
    assert np.isfinite(whole[0]).all() and np.isfinite(whole[1]).all()
    for every, budget in ((7, None), (whole[2] + 1, None), (64, 1)):
        runs.clear()
        if budget:  # no room for the record: checkpoints
            monkeypatch.setattr(_autodiff, "CHECKPOINT_STORE_BUDGET", budget)
        other = gradients(every)
        assert [r[0] for r in runs] == [whole[2] // every + 1]
        assert every > 64 or runs[0][1] is None
        np.testing.assert_array_equal(other[0], whole[0])
        np.testing.assert_array_equal(other[1], whole[1])
