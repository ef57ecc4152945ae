"""Quotients by a pivot taken through its reciprocal, bit for bit the oracle's
divisions: at ordinary magnitudes and at those where the reciprocal's way does
not hold (subnormal floats; doubles near the ends of their exponents), in some
trajectories of a wavefront and not in others, in the unrolled dense solve, the
row-a-lane solve and the register adjoint."""

import numpy as np
import pytest

from menodax_amd import rodas5P
from oracle import oracle as O
from tests import systems as S
from tests.test_gpu_parity import _pivoting_blocks, _same

pytestmark = pytest.mark.gpu

SCALES = {"ordinary": [1.0], "small": [1e-39, 1.0, 1e-44, 1e-42],
          "smallest": [1e-290, 1.0, 1e-305, 1e-322, 1e-250], "largest": [1e60, 1e150, 1.0, 1e140]}


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("scales", SCALES)
@pytest.mark.parametrize("n", [4, 16, 20, 34])
def test_solves(n, scales, lu):
    fn, system, y0, p = _pivoting_blocks(n, 70, seed=n)
    y0 = y0 * np.resize(SCALES[scales], 70)[:, None]
    t = np.linspace(0.0, 0.05, 4)
    run = dict(rtol=1e-6, atol=1e-8, first_step=1e-3, max_steps=300, lu_precision=lu)
    hist, st = rodas5P.solve(fn, y0, t, p, return_stats=True,
                             placement="wave" if n > 16 else None, **run)
    ref, rst = O.rodas5p(system, y0, t, p, **run)
    reached = ~np.isnan(hist)
    np.testing.assert_array_equal(hist[reached], ref[reached])
    for k in rst:
        np.testing.assert_array_equal(st[k], rst[k])
    if scales != "largest":
        assert reached.all()


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("scale", [1.0, 1e-300, 1e290])
def test_the_register_adjoint(lu, scale):
    fn, _, y0, p = _pivoting_blocks(4, 70, seed=4)
    t = np.linspace(0.0, 0.05, 4)
    g = np.random.default_rng(0).normal(size=(70, 4, 4)) * scale
    run = dict(rtol=1e-6, atol=1e-8, lu_precision=lu)
    got = rodas5P.adjoint_gradients(fn, y0, t, p, g, **run)
    ref = rodas5P.adjoint_gradients(fn, y0, t, p, g, placement="rolled", **run)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all() and (a != 0).any()
        np.testing.assert_array_equal(a, b)
