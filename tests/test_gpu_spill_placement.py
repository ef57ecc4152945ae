"""Kernels whose spills were misplaced give what the same step gives in another
placement, bit for bit: a joint solve under a three-term controller, and the
rolled Tsit5 step of a 19-variable system in workgroups of 64, 32 and 16."""

import numpy as np
import pytest

from menodax_amd import _kernels as K, rodas5P
from tests import systems as S
from tests.test_spill_placement import coupled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("control", [True, False])
@pytest.mark.parametrize("wrt_params", [True, False])
def test_joint_solve_with_a_three_term_controller(lu, control, wrt_params):
    y0, p = S.robertson_lognormal_ensemble(127, seed=5)
    t = np.array([0.0, 0.25, 0.25, 0.37, 1.3, 1.9])

    def solve(placement):
        return rodas5P.solve_sensitivities(
            S.robertson, y0, t, p, wrt_y0=True, wrt_params=wrt_params, sens_error_control=control,
            placement=placement, lu_precision=lu, return_stats=True, rtol=1e-6, atol=1e-9,
            first_step=0.5, max_steps=400, pcoeff=0.2, icoeff=0.6, dcoeff=0.1)

    got, ref = solve("registers"), solve("rolled")
    assert ref[2]["accepted_steps"].min() > 0 and ref[2]["loop_steps"].max() < 400
    for k in ref[2]:
        np.testing.assert_array_equal(got[2][k], ref[2][k])
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])


@pytest.mark.parametrize("n", [17, 19, 24])
def test_rolled_tsit5_in_every_placement(n):
    import torch

    fn = coupled(n)
    rng = np.random.default_rng(n)
    dev = torch.device("cuda")
    y0 = torch.as_tensor(rng.uniform(-1.0, 1.0, (200, n)), device=dev)
    p = torch.as_tensor(10.0 ** rng.uniform(-1.0, 1.0, (200, 4)), device=dev)
    t = torch.as_tensor([0.0, 0.4, 0.4, 0.4 + 1e-13, 1.4, 1.54, 1.85], dtype=torch.float64,
                        device=dev)
    runs = []
    for placement, block in (("rolled", 64), ("lds", 64), ("lds", 32), ("lds", 16), (None, 64),
                             ("team", 64)):
        built = K.tsit5_kernel(fn, n, 4, K.Tsit5Options(placement=placement,
                                                        trajectories_per_block=block))
        out = rodas5P.launch(built, y0, t, p, 200, dt0=1e-4, rtol=1e-6, atol=1e-9, max_steps=400)
        torch.cuda.synchronize()
        runs.append((out.hist.cpu().numpy(), out.accepted.cpu().numpy(), out.loop.cpu().numpy()))
    assert np.isfinite(runs[0][0]).all() and runs[0][2].max() < 400
    for other in runs[1:]:
        for a, b in zip(other, runs[0]):
            np.testing.assert_array_equal(a, b)
