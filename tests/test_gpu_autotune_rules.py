"""The autotuner's options against what ``solve`` takes by its size rules, which
none of its candidates may be: a team, eight lanes a trajectory."""

import numpy as np
import pytest

from menodax_amd import autotune, rodas5P
from tests import systems as S

pytestmark = pytest.mark.gpu

DEFAULTS = {"placement": None, "trajectories_per_block": None, "refill": None,
            "tableau_in_registers": None}


def test_a_team_two_times_as_fast_as_any_candidate_is_left_to_the_rules():
    fn, mask = S.vdp_lattice(12)[0], S.vdp_sparsity(12)
    y0, p = S.vdp_scenario(12, 1000, 42, divergence=0.25)
    kw = dict(first_step=1e-4, rtol=1e-6, atol=1e-8, lu_precision="fp32", sparsity=mask)
    opts = autotune.tuned_options(fn, y0, S.VDP_TIMES, p, blocks=(64,), reps=3, **kw)
    assert opts == DEFAULTS
    np.testing.assert_array_equal(rodas5P.solve(fn, y0, S.VDP_TIMES, p, **opts, **kw),
                                  rodas5P.solve(fn, y0, S.VDP_TIMES, p, placement="lds", **kw))


@pytest.mark.parametrize("sample", [None, 512])
def test_the_faster_of_the_two_is_what_the_options_say(monkeypatch, sample):
    """Both outcomes, whatever the clock says."""
    y0, p = S.robertson_lognormal_ensemble(1024, seed=3)
    t = S.robertson_benchmark_times()
    kw = dict(rtol=1e-6, atol=1e-8, lu_precision="fp32")
    best, table, own = autotune._measured(S.robertson, y0, t, p, blocks=(64,), sample=sample, **kw)
    assert own > 0 and best.seconds == min(c.seconds for c in table)
    for seconds in (best.seconds / 2, best.seconds * 2):
        monkeypatch.setattr(autotune, "_measured", lambda *a, **k: (best, table, seconds))
        opts = autotune.tuned_options(S.robertson, y0, t, p)
        assert (opts == DEFAULTS) == (seconds < best.seconds)
        assert seconds < best.seconds or opts["trajectories_per_block"] == best.trajectories_per_block
