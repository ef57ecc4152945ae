"""Joint sensitivity solves of a team against the rolled one-lane kernel, bit
for bit: one direction, several, and as many as put one trajectory in a
workgroup; ensembles that leave its last trajectories out; every error control
and weights; and the row-a-lane wave kernel's row counts against the oracle
where the factorisation swaps rows."""

import numpy as np
import pytest

from menodax_amd import _kernels as K, rodas5P
from menodax_amd._sensitivity import SensitivitySpec
from menodax_amd._sparsity import normalize_sparsity
from oracle import oracle as O
from tests import systems as S
from tests.test_gpu_parity import _pivoting_blocks, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_osc, traj, wrt_y0, wrt_params, control", [
    (9, 65, False, True, True), (12, 7, False, True, False), (32, 33, False, True, True),
    (9, 4, True, False, True), (10, 5, True, True, False)])
def test_a_team_changes_no_bit(n_osc, traj, wrt_y0, wrt_params, control):
    n, mask = 2 * n_osc, S.vdp_sparsity(n_osc)
    fn, _ = S.vdp_lattice(n_osc)
    spec = SensitivitySpec(n, 1, wrt_y0, wrt_params, control, None)
    assert K.rodas5p_team(fn, n, 1, K.KernelOptions(sparsity=normalize_sparsity(mask, n),
                                                    sens=spec))
    y0, p = S.vdp_scenario(n_osc, traj, 42, divergence=0.25)
    w = np.random.default_rng(0).uniform(0.5, 2.0, size=(traj, n))
    for weights, max_steps in ((None, 100000), (w if n_osc == 9 else None, 20)):
        run = dict(first_step=1e-4, rtol=1e-6, atol=1e-8, sparsity=mask, wrt_y0=wrt_y0,
                   wrt_params=wrt_params, sens_error_control=control, error_weights=weights,
                   max_steps=max_steps)
        got = rodas5P.solve_sensitivities(fn, y0, S.VDP_TIMES, p, **run)
        want = rodas5P.solve_sensitivities(fn, y0, S.VDP_TIMES, p, placement="rolled", **run)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("n, traj", [(18, 1), (32, 5), (34, 70), (50, 3), (64, 9)])
def test_rows_a_lane_pivot_as_the_sequential_scan(n, traj, lu):
    fn, system, y0, p = _pivoting_blocks(n, traj, seed=n)
    t = np.linspace(0.0, 0.05, 5)
    run = dict(rtol=1e-6, atol=1e-8, lu_precision=lu)
    hist, st = rodas5P.solve(fn, y0, t, p, placement="wave", return_stats=True, **run)
    _same(hist, st, *O.rodas5p(system, y0, t, p, **run))


def test_rows_a_lane_registered_as_one_wavefront_a_workgroup():
    """A handle made with MDX_KERNEL_WAVE alone launches a workgroup of 64 lanes
    a trajectory: the same bits."""
    import dataclasses

    import torch

    from menodax_amd import _runtime

    fn, _, y0, p = _pivoting_blocks(20, 9)
    options = K.KernelOptions(placement="wave")
    built = K.rodas5p_kernel(fn, 20, 30, options)
    source, _ = K.rodas5p_source(fn, 20, 30, options)
    handle = _runtime.kernel_create(_runtime.code_object(source, "wave.hip"), "mdx_rodas5p", 64,
                                    _runtime.KERNEL_UNIT_WEIGHTS | _runtime.KERNEL_WAVE)
    dev = torch.device("cuda")
    args = [torch.tensor(x, device=dev) for x in (y0, np.linspace(0.0, 0.05, 4), p)]
    run = dict(dt0=0.0, rtol=1e-6, atol=1e-8, max_steps=1000)
    one, four = (rodas5P.launch(b, *args, 9, **run).ensemble_view()
                 for b in (dataclasses.replace(built, plain=handle), built))
    assert torch.isfinite(four).all() and torch.equal(one, four)
