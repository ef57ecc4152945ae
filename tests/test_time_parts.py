"""A right-hand side whose time part is computed apart: the emitted parts,
compiled for the CPU, against the undivided code, bit for bit, and the rule."""

import ctypes
import math
import subprocess

import numpy as np
import pytest

from menodax_amd import _codegen as C, _kernels as K
from menodax_amd._sparsity import dense_jacobian
from tests import systems as S


def forced(y, t, p):
    # a comparison of times under a state-dependent choice, an output that
    # never reads the state, values of the parameters alone, a time part the
    # Jacobian starts from
    drive = math.exp(-p[0] * t) * math.sin(t) ** 2 + math.cos(2.0 * t) / (1.0 + t ** 2)
    gate = (t > 1.0) * y[0]
    rate = 10.0 ** p[1]
    return (gate - rate * y[0] * drive, drive / rate, math.sqrt(1.0 + t) * y[0] * y[2] - y[2] ** 2)


HARNESS = """
#include <cmath>
using namespace std;
#define __device__
#define __forceinline__ inline
namespace mdx { template <class T> struct lu_elem; template <> struct lu_elem<double*> { typedef double type; }; }
namespace whole { %s }
namespace part { %s }
struct P { const double* v; double x[8]; double operator[](int i) const { return v[i]; } };
struct TP { const double* v; double operator()(int m) const { return v[m]; } };
extern "C" void run(const double* y, double t, const double* pv, double* a, double* b) {
  P p; p.v = pv;
  whole::rhs(y, t, p, a);
  whole::neg_jac(y, t, p, a + %d, a + %d);
  double tp[16];
  part::param_part(p, p.x);
  part::time_part(t, p, tp);
  part::rhs(y, t, p, TP{tp}, b);
  part::neg_jac(y, t, p, TP{tp}, b + %d, b + %d);
}
"""


@pytest.mark.parametrize("fn, n, n_params, t", [(S.bbn, 4, 2, (0.13, 3.0, 90.0)),
                                                (forced, 3, 2, (0.0, 1.0, 2.5))])
def test_the_parts_compute_what_the_whole_does(fn, n, n_params, t, tmp_path):
    tr = C.trace(fn, n, n_params)
    st = dense_jacobian(n)
    kw = dict(colour=st.colour, n_colours=st.n_colours, store=st.stores())
    source, parts = C.generate_in_parts(tr, **kw)
    stage = source[source.index("rhs(const YA&"):source.index("neg_jac(const YA&")]
    assert not any(f"{call}(" in stage for call in ("exp", "pow", "sin", "cos", "sqrt"))
    cpp = tmp_path / "parts.cpp"
    cpp.write_text(HARNESS % (C.generate(tr, **kw).source, source, n, n + n * n, n, n + n * n))
    lib = tmp_path / "parts.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-o", lib, cpp], check=True)
    run = ctypes.CDLL(str(lib)).run
    rng = np.random.default_rng(0)
    ptr = lambda x: x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))  # noqa: E731
    for time in t:
        y = rng.uniform(0.1, 1.0, n)
        p = np.array([1.2, 0.4]) if fn is forced else np.array([0.78, 3.044])
        a, b = np.full((2, 2 * n + n * n), np.nan)
        run(ptr(y), ctypes.c_double(time), ptr(p), ptr(a), ptr(b))
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a.view(np.int64), b.view(np.int64))


def test_the_rule():
    o = K.KernelOptions()
    assert K.time_lanes(S.bbn, 4, 2, o, 8192, 256) == K.TIME_LANES
    assert K.time_lanes(S.bbn, 4, 2, o, 8193, 256) == 1  # a SIMD would hold two wavefronts
    assert K.time_lanes(S.robertson, 3, 3, o, 64, 256) == 1  # does not read the time
    for kw in (dict(placement="rolled"), dict(max_registers=128), dict(save_hook=lambda *a: None)):
        assert K.time_lanes(S.bbn, 4, 2, K.KernelOptions(**kw), 64, 256) == 1
    for kw in (dict(trajectories_per_block=4), dict(trajectories_per_block=256),
               dict(placement="rolled")):
        with pytest.raises(ValueError):
            K.rodas5p_source(S.bbn, 4, 2, K.KernelOptions(lanes=8, **kw))
    with pytest.raises(ValueError):
        K.rodas5p_source(S.robertson, 3, 3, K.KernelOptions(lanes=8))
