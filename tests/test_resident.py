"""The bound on an unrolled kernel's registers: taken where it costs a few
spilled ones, not where a right-hand side needs many more (compiled here, read
from the code objects)."""

import math

import pytest

from menodax_amd import _kernels as K, _runtime
from tests import systems as S


def with_calls(y, t, p):
    e, s = math.exp(-y[0] * y[0]), math.sin(y[1] * p[0])
    q, r = math.sqrt(1.0 + y[2] * y[2]), (1.0 + y[0] * y[0]) ** 1.5
    return (-p[0] * y[0] * e + p[1] * s / q, p[0] * e - p[1] * y[1] * q - r * 0.1,
            s * e / r - 0.3 * y[2] * q)


def dense6(y, t, p):
    return tuple(
        sum((0.1 * (i - j) * y[j] * y[(i + j) % 6] for j in range(6) if j != i),
            -(1.0 + p[0] * (i + 1)) * y[i]) for i in range(6))


def _registers(fn, n, n_p, **kw):
    source, d = K.rodas5p_source(fn, n, n_p, K.KernelOptions(**kw))
    _, code = K.bounded_code(source, "test_resident.hip", d["resident"])
    kernels = _runtime.kernel_registers(code)
    assert {"mdx_rodas5p", "mdx_rodas5p_refill"} <= set(kernels)
    return [kernels[k] for k in ("mdx_rodas5p", "mdx_rodas5p_refill")]


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("tableau", [False, True])
def test_robertson_keeps_the_wavefronts_its_ensembles_count_on(lu, tableau):
    for k in _registers(S.robertson, 3, 3, lu_precision=lu, tableau_in_registers=tableau):
        assert k["vgprs"] <= (256 if tableau else 168)
        assert k["spills"] <= K.RESIDENT_MAX_SPILLS


def test_an_ensemble_of_two_wavefronts_a_simd_is_not_bounded_to_three():
    plain = _registers(S.robertson, 3, 3, lu_precision="fp64", resident=2)
    assert all(168 < k["vgprs"] <= 256 and k["spills"] == 0 for k in plain)


@pytest.mark.parametrize("fn, n, n_p, kw", [
    (with_calls, 3, 2, dict(lu_precision="fp32")),
    (with_calls, 3, 2, dict(lu_precision="fp64")),
    (with_calls, 3, 2, dict(lu_precision="fp32", tableau_in_registers=True)),
    (with_calls, 3, 2, dict(lu_precision="fp64", tableau_in_registers=True)),
    (dense6, 6, 1, dict(lu_precision="fp64")),
    (S.robertson, 3, 3, dict(lu_refine=True, tableau_in_registers=True)),
    (S.damped_oscillator, 2, 2, dict(save_hook=S.energy_hook, hook_size=33, hook_n_save=33))])
def test_a_kernel_that_needs_more_spills_nothing_to_memory(fn, n, n_p, kw):
    assert all(k["scratch"] == 0 for k in _registers(fn, n, n_p, **kw))


@pytest.mark.parametrize("sens", [False, True])
def test_the_wave_placement_keeps_to_the_callers_registers(sens):
    """The cap counts one of the register file's two halves."""
    from menodax_amd._sensitivity import SensitivitySpec

    n = 24
    source, _ = K.rodas5p_source(S.vdp_lattice(12)[0], n, 1, K.KernelOptions(
        placement="wave", max_registers=48,
        sens=SensitivitySpec(n, 1, False, True) if sens else None))
    code = _runtime.code_object(source, "test_resident_wave.hip")
    assert _runtime.kernel_registers(code)["mdx_rodas5p"]["vgprs"] <= 96
