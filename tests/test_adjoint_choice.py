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


@pytest.mark.parametrize("ckpt_every, placement", [(64, "team"), (16, "lds"), (64, None)])
def test_a_gradient_builds_the_adjoint_it_expects_to_run_and_no_other(monkeypatch, ckpt_every,
                                                                      placement):
    """Compiling an adjoint takes seconds: the checkpoints' kernel of a system
    whose records fit waits until it is wanted."""
    import types

    import torch

    from menodax_amd import _autodiff

    built = []

    def adjoint_kernel(ode_fn, n_vars, n_params, options):
        built.append(options)
        return types.SimpleNamespace(options=options, extra={})

    monkeypatch.setattr(K, "rodas5p_adjoint_kernel", adjoint_kernel)
    monkeypatch.setattr(K, "rodas5p_kernel", lambda *a: None)
    monkeypatch.setattr(_common, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(rodas5P, "_tableau", lambda *a: False)
    monkeypatch.setattr(rodas5P, "_sized", lambda options, *a: options)
    jobs = []
    monkeypatch.setattr(_autodiff, "adjoint_solve",
                        lambda job, y, p: (jobs.append(job) or y, (None, None, None)))
    fn, n, options = _chain(10 if placement else 1, lu_precision="fp64")
    y0 = torch.ones((500, n), dtype=torch.float64, requires_grad=True)
    rodas5P.solve(fn, y0, [0.0, 1.0], torch.ones((500, 1), dtype=torch.float64), adjoint=True,
                  ckpt_every=ckpt_every, lu_precision="fp64",
                  sparsity=S.vdp_sparsity(10, wrap=False) if placement else None)
    assert [(o.placement, o.adjoint_keep) for o in built] == [(placement, placement is None)]
    # the other one when it is asked for
    (job,) = jobs
    checkpoints = job.adjoint().options
    assert checkpoints.placement == ("lds" if placement else None) and not checkpoints.adjoint_keep
