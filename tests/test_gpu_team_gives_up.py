"""A team launch that does not get all its workgroups: the pass is finished by
launches, and the solves after it are unharmed.  The starved launch has one
workgroup too few for its largest problem and the error flag set that a wait
looks at, so each wait ends after some thousand polls and the kernel returns.
"""
import numpy as np
import pytest

import amie_gpu as ag
import configs
from test_gpu_team import grids

pytestmark = pytest.mark.gpu

CASES = {
    "one": lambda: grids([60]),
    "several_and_single": lambda: grids([60, 45, 9]),
    "over_64_tiles": lambda: grids([150]),
    "three_loads": lambda: [configs.rve(n, 40 + n, 0.3) for n in (60, 33)],
    "tet4": lambda: [configs.config3(13, seed=8)],
}


@pytest.mark.parametrize("precision", [ag.FP64, ag.MIXED_FIX48])
@pytest.mark.parametrize("use_x0", [0, 1])
@pytest.mark.parametrize("case", list(CASES))
def test_pass_is_finished_by_launches(case, use_x0, precision):
    """Nothing of the starved launch's first problem reaches its iterate, so
    the launches' results are those of a launch-path solve bit for bit; the
    single-workgroup problems of the batch may have ended by themselves."""
    probs = CASES[case]()
    ctx = ag.Context(0)
    B = ag.Batch(ctx, probs)

    def solve(use):
        for k, p in enumerate(probs):
            B.set_solution(np.tile(1e-5 * np.sin(np.arange(p.ndof)), p.nrhs), k)
        B.set_team(use, 1)
        st = B.solve(precision=precision, rtol=1e-10, use_x0=use_x0)
        return st, [B.solution(k).copy() for k in range(len(probs))], B.team_info()

    st, ref, info = solve(ag.TEAM_NEVER)
    assert st["status"] == 0 and info["team_passes"] == 0
    for use, team, gave_up in ((ag.TEAM_STARVED, 1, 1), (ag.TEAM_ALWAYS, 1, 0), (ag.TEAM_STARVED, 1, 1),
                               (ag.TEAM_NEVER, 0, 0)):
        print(case, precision, use_x0, use, flush=True)
        got, x, info = solve(use)
        assert (info["passes"], info["team_passes"], info["gave_up"]) == (1, team, gave_up)
        assert got["status"] == 0 and got["iterations_sum"] == st["iterations_sum"]
        for a, b in zip(x, ref):
            np.testing.assert_array_equal(a, b)
    # from then on this batch keeps to launches, until it is told otherwise
    solve(ag.TEAM_STARVED)
    for _ in range(2):
        B.solve(precision=precision, rtol=1e-10)
        assert B.team_info()["team_passes"] == 0
    B.set_team(ag.TEAM_ALWAYS)
    B.solve(precision=precision, rtol=1e-10)
    assert B.team_info()["gave_up"] == 0 and B.team_info()["team_passes"] == 1
    B.close()
    ctx.close()
