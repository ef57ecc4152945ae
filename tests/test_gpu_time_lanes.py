"""Eight lanes a trajectory, sharing out the right-hand side's time part,
against one lane, bit for bit: ensembles that do and do not fill a wavefront
and a workgroup, saves inside the interval, weights, a step budget, refinement
and an FP64 LU."""

import numpy as np
import pytest

from menodax_amd import _kernels as K, rodas5P
from tests import systems as S
from tests.test_time_parts import forced

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 9, 70, 2500, 8192])
@pytest.mark.parametrize("kw", [
    dict(lu_precision="fp32"), dict(lu_precision="fp64", max_steps=40),
    dict(lu_precision="fp32", lu_refine=True, rtol=1e-6)], ids=["fp32", "budget", "refined"])
@pytest.mark.parametrize("fn", [S.bbn, forced], ids=["bbn", "forced"])
def test_the_same_bits(fn, n, kw, monkeypatch):
    rng = np.random.default_rng(n)
    if fn is forced:
        y0, p = rng.uniform(0.5, 1.5, (n, 3)), rng.uniform(0.1, 1.0, (n, 2))
        t, run = np.array([0.0, 0.3, 0.31, 2.0]), dict(dict(rtol=1e-5, atol=1e-8), **kw)
    else:
        y0, p = np.tile([0.85, 0.15, 0.0, 0.0], (n, 1)), np.column_stack(
            [rng.uniform(0.0, 1.5, n), rng.uniform(2.5, 3.5, n)])
        t = np.array([0.1293, 1.0, 60.0, 129.3])
        run = dict(dict(rtol=1e-4, atol=1e-9, first_step=0.1, max_steps=256), **kw)
    w = None if n % 2 else rng.uniform(0.5, 2.0, y0.shape)
    assert K.time_lanes(fn, *y0.shape[1:], 2, K.KernelOptions(), n, 256) == K.TIME_LANES
    got, st = rodas5P.solve(fn, y0, t, p, error_weights=w, return_stats=True, **run)
    monkeypatch.setattr(K, "time_lanes", lambda *a: 1)
    ref, rst = rodas5P.solve(fn, y0, t, p, error_weights=w, return_stats=True, **run)
    np.testing.assert_array_equal(got, ref)
    for k in rst:
        np.testing.assert_array_equal(st[k], rst[k])
