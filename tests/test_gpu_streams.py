"""A solve and its gradients on a stream of the caller's: ordered after what the
current stream still has to do to the inputs, its tensors not given out again
while it runs, and its results waited for where they are read."""

import numpy as np
import pytest

from menodax_amd import rodas5P, tsit5
from tests import systems as S

pytestmark = pytest.mark.gpu


@pytest.fixture()
def busy():
    """A side stream, and the current stream with some milliseconds still to run."""
    import torch

    side = torch.cuda.Stream()

    def fill():
        x = torch.ones((4096, 4096), device="cuda")
        for _ in range(20):
            x = (x @ x).clamp_(-1.0, 1.0)

    return side, fill


@pytest.mark.parametrize("module", [rodas5P, tsit5])
def test_solves(module, busy):
    import torch

    side, fill = busy
    y0, p = S.lorenz_rho_ensemble(4096)
    t = np.linspace(0.0, 1.0, 20)
    ref = module.solve(S.lorenz, y0, t, p)
    y, q = torch.as_tensor(y0, device="cuda"), torch.as_tensor(p, device="cuda")
    fill()
    got = module.solve(S.lorenz, y * 1.0, torch.as_tensor(t), q * 1.0, stream=side)
    junk = [torch.full((4096, 3), 7.0, device="cuda", dtype=torch.float64) for _ in range(8)]
    side.synchronize()
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    assert all(float(x[0, 0]) == 7.0 for x in junk)
    fill()
    np.testing.assert_array_equal(module.solve(S.lorenz, y0, t, p, stream=side), ref)


@pytest.mark.parametrize("n_osc", [1, 10])
@pytest.mark.parametrize("ckpt_every", [16, 64])
def test_gradients(n_osc, ckpt_every, busy):
    import torch

    side, fill = busy
    fn, _ = S.vdp_lattice(n_osc, mu=1.0, d=0.1, wrap=False)
    y0, p = S.vdp_scenario(n_osc, 70, 3, divergence=0.9)
    t = np.linspace(0.0, 3.0, 6)
    kw = dict(rtol=1e-8, atol=1e-10, lu_precision="fp64",
              sparsity=S.vdp_sparsity(n_osc, wrap=False) if n_osc > 1 else None)
    g = np.random.default_rng(0).normal(size=(70, 6, 2 * n_osc))
    ref = rodas5P.adjoint_gradients(fn, y0, t, p, g, ckpt_every=ckpt_every, **kw)
    fill()
    got = rodas5P.adjoint_gradients(fn, y0, t, p, g, ckpt_every=ckpt_every, stream=side, **kw)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])
    y = torch.tensor(y0, device="cuda", requires_grad=True)
    q = torch.tensor(p, device="cuda", requires_grad=True)
    fill()
    hist = rodas5P.solve(fn, y, t, q, adjoint=True, ckpt_every=ckpt_every, stream=side, **kw)
    (hist * torch.as_tensor(g, device="cuda")).sum().backward()
    np.testing.assert_array_equal(y.grad.cpu().numpy(), ref[0])
    np.testing.assert_array_equal(q.grad.cpu().numpy(), ref[1])


def test_forward_sensitivities(busy):
    side, fill = busy
    y0, p = S.robertson_lognormal_ensemble(256, seed=1)
    t = S.robertson_benchmark_times()
    ref = rodas5P.solve_sensitivities(S.robertson, y0, t, p, rtol=1e-6, atol=1e-8)
    fill()
    got = rodas5P.solve_sensitivities(S.robertson, y0, t, p, rtol=1e-6, atol=1e-8, stream=side)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])
