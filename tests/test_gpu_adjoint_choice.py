"""Adjoint gradients where the caller chooses the forward solve's placement or
the store's size: the same bits whichever kernel they bring in."""

import numpy as np
import pytest

from menodax_amd import rodas5P
from tests import systems as S

pytestmark = pytest.mark.gpu


def _chain_problem(n_traj=70):
    fn, _ = S.vdp_lattice(10, mu=1.0, d=0.1, wrap=False)
    y0, mu = S.vdp_scenario(10, n_traj, 3, divergence=0.9)
    t = np.array([0.0, 0.5, 0.500001, 2.9, 3.0])
    g = np.random.default_rng(0).normal(size=(n_traj, t.size, 20))
    kw = dict(rtol=1e-8, atol=1e-10, lu_precision="fp64", sparsity=S.vdp_sparsity(10, wrap=False))
    return fn, y0, mu, t, g, kw


@pytest.mark.parametrize("ckpt_every", [16, 64])
def test_the_team_placement_asked_for(ckpt_every):
    """More steps than a checkpoint interval, with and without room for every
    step's record (a ckpt_every under the default asks for checkpoints)."""
    import torch

    fn, y0, mu, t, g, kw = _chain_problem()
    dev = torch.device("cuda")

    def gradients(**place):
        y = torch.tensor(y0, device=dev, requires_grad=True)
        p = torch.tensor(mu, device=dev, requires_grad=True)
        hist, st = rodas5P.solve(fn, y, t, p, adjoint=True, ckpt_every=ckpt_every,
                                 return_stats=True, **place, **kw)
        assert int(st["accepted_steps"].max()) > ckpt_every
        (hist * torch.as_tensor(g, device=dev)).sum().backward()
        return y.grad.cpu().numpy(), p.grad.cpu().numpy()

    ref = gradients()
    got = gradients(placement="team")
    direct = rodas5P.adjoint_gradients(fn, y0, t, mu, g, ckpt_every=ckpt_every, placement="team", **kw)
    assert np.isfinite(ref[0]).all() and np.isfinite(ref[1]).all()
    for other in (got, direct):
        np.testing.assert_array_equal(other[0], ref[0])
        np.testing.assert_array_equal(other[1], ref[1])
