"""The size rules and row tables of the team placement (a trajectory's rows
shared out over a workgroup's wavefronts), on the host."""

import math

import numpy as np
import pytest

from menodax_amd import _codegen, _kernels as K
from menodax_amd._sparsity import normalize_sparsity
from tests import systems as S


def _sparse(mask, **kw):
    return K.KernelOptions(sparsity=normalize_sparsity(mask, len(mask)), **kw)


@pytest.mark.parametrize("waves, first", [(8, 0), (8, 1), (4, 1), (16, 0)])
@pytest.mark.parametrize("n", [17, 24, 50, 63])
def test_every_row_has_one_slot(n, waves, first):
    fn, _, _ = S.arrow_system(n)
    traced = _codegen.trace(fn, n, S.arrow_n_params(n))
    team = _codegen.deal_rows(traced, waves, first)
    assert sorted(v for vs in team.rows for v in vs) == list(range(n))
    assert all(vs == () for vs in team.rows[:first])
    assert team.per_wave == math.ceil(n / (waves - first))
    assert max(len(vs) for vs in team.rows) <= team.per_wave
    slots = team.slot_of
    assert len(set(slots)) == n and 0 <= min(slots)
    assert max(slots) < (waves - first) * team.per_wave
    space = {}
    for line in team.tables().splitlines():
        name, values = line.split("int ")[1].split(" = ")
        space[name.split("[")[0]] = [int(v) for v in values.strip("{};").split(",")]
    assert space["SLOT_OF"] == slots
    assert [space["ROW_OF"][s] for s in slots] == list(range(n))
    assert space["ROW_OF"].count(-1) == (waves - first) * team.per_wave - n
    # every wavefront's branch writes all of its slots
    src = _codegen.generate_rhs_rows(traced, team)
    for w in range(waves):
        body = src.split(f"case {w}:")[1].split("break;")[0]
        assert [f"out[{j}]" in body for j in range(team.per_wave)] == [True] * team.per_wave


def test_the_rodas5p_rule_leaves_out_what_a_team_cannot_step():
    ring, mask = S.vdp_lattice(12)[0], S.vdp_sparsity(12)
    assert K.rodas5p_team(ring, 24, 1, _sparse(mask))
    assert K.rodas5p_team(ring, 24, 1, _sparse(mask, lu_precision="fp64"))
    for n_osc in (8, 33):  # 16 and 66 variables: the unrolled step, and too many rows
        assert not K.rodas5p_team(S.vdp_lattice(n_osc)[0], 2 * n_osc, 1, _sparse(S.vdp_sparsity(n_osc)))
    assert K.rodas5p_team(S.vdp_lattice(9)[0], 18, 1, _sparse(S.vdp_sparsity(9)))
    assert K.rodas5p_team(S.vdp_lattice(32)[0], 64, 1, _sparse(S.vdp_sparsity(32)))
    assert not K.rodas5p_team(ring, 24, 1, K.KernelOptions())  # dense
    for kw in (dict(placement="lds"), dict(lu_refine=True), dict(max_registers=128),
               dict(save_hook=lambda *a: None, hook_size=1)):
        assert not K.rodas5p_team(ring, 24, 1, _sparse(mask, **kw))

    def forced(y, t, p):
        f = ring(y, t, p)
        return (f[0] + 0.1 * t,) + tuple(f[1:])

    assert not K.rodas5p_team(forced, 24, 1, _sparse(mask))  # reads t
    with pytest.raises(ValueError, match="team placement"):
        K.rodas5p_source(forced, 24, 1, _sparse(mask, placement="team"))
    bordered, bmask, _ = S.bordered_system()
    assert not K.rodas5p_team(bordered, len(bmask), len(bmask), _sparse(bmask))

    def shared(y, t, p):
        # one product that every row needs: dealing the rows out repeats it
        s = y[0]
        for j in range(1, 24):
            s = s * y[j] + y[j] * y[j - 1]
        return tuple(s - y[j] for j in range(24))

    assert not K.rodas5p_team(shared, 24, 1, _sparse(np.ones((24, 24), dtype=bool)))
    assert not K.tsit5_team(None, 24, 1, shared) and K.tsit5_team(None, 24, 1, ring)


def test_the_tsit5_rule():
    def team(requested, n, n_params=1):
        return K.tsit5_team(requested, n, n_params, S.vdp_lattice(n // 2, mu=1.0)[0])

    assert not team(None, 16)
    assert team(None, 18) and team(None, 64)
    assert not team(None, 66)
    assert not team(64, 32)  # the caller's workgroup
    # a parameter row too wide for the LDS next to the exchange buffers
    assert team(None, 64, 100) and not team(None, 64, 200)
    with pytest.raises(ValueError, match="bytes of LDS"):
        K.tsit5_source(S.vdp_lattice(32, mu=1.0)[0], 64, 300, K.Tsit5Options(placement="team"))


@pytest.mark.parametrize("n, expect", [(1, 64), (64 * 256, 64), (64 * 256 + 1, 128),
                                       (128 * 256, 128), (128 * 256 + 1, 256), (256 * 256, 256),
                                       (256 * 256 + 1, 64), (10**6, 64)])
def test_an_unrolled_solves_workgroup_covers_a_compute_unit(n, expect):
    assert K.register_block(n, 256) == expect
