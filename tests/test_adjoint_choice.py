"""Which adjoint kernel a solve takes, on the host: the one that keeps
checkpoints and, where every step's record fits, the one that needs no
checkpoints."""

import pytest

from menodax_amd import _common, _kernels as K, rodas5P
from menodax_amd._sparsity import normalize_sparsity
from tests import systems as S


@pytest.fixture(autouse=True)
def compute_units(monkeypatch):
    monkeypatch.setattr(_common, "n_cu", lambda: 256)


def _chain(n_osc, **kw):
    n = 2 * n_osc
    fn, _ = S.vdp_lattice(n_osc, mu=1.0, d=0.1, wrap=False)
    return fn, n, K.KernelOptions(sparsity=normalize_sparsity(S.vdp_sparsity(n_osc, wrap=False), n),
                                  **kw)


@pytest.mark.parametrize("lu", ["fp32", "fp64"])
@pytest.mark.parametrize("n_osc, block", [(3, None), (5, None), (10, None), (10, 16)])
def test_a_team_solves_checkpoints_are_another_kernels(n_osc, block, lu):
    """The team's adjoint knows one checkpoint only: a caller's placement="team"
    must not make it the kernel of the checkpoints."""
    fn, n, options = _chain(n_osc, lu_precision=lu, placement="team",
                            trajectories_per_block=block or 64)
    chosen = rodas5P._adjoint_options(options, n, 500, block)
    source, details = K.rodas5p_source(fn, n, 1, chosen, adjoint=True)
    assert chosen.placement != "team" and "MDX_TEAM" not in source
    # the rest is as without the caller's placement
    _, _, free = _chain(n_osc, lu_precision=lu, trajectories_per_block=block or 64)
    assert chosen == rodas5P._adjoint_options(free, n, 500, block)
    whole = rodas5P._whole_adjoint(options, fn, n, 1, 500, block)
    assert bool(whole) == (block is None and n > K.ADJOINT_UNROLLED_MAX_VARS)
