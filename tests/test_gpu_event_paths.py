"""How the solves of an event-driven damage step run."""
import numpy as np
import pytest

import amie_gpu as ag
import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [(12, ag.FP64), (12, ag.MIXED_FIX48), (40, ag.FP64)])
def test_event_step_solves_as_one_launch(n, precision):
    """Also with time_kernels, which a step has no field for: a team of one
    workgroup and of several, the same damage and displacements."""
    prob, dofs, nfix, crit, maz, radius = configs.event_square(n)
    vals = np.concatenate([np.zeros(nfix), np.full(len(dofs) - nfix, 0.8e-4)])
    ctx = ag.Context(0)
    out = []
    for time_kernels in (0, 1):
        B = ag.Batch(ctx, [prob])
        B.set_bc_values(dofs, vals)
        st = B.event_step(crit, maz, radius, precision=precision, rtol=1e-12, time_kernels=time_kernels)
        info = B.team_info()
        assert st["status"] == 0 and info["team_passes"] == info["passes"] == 1, (st, info)
        assert (info["workgroups"] > 1) == (n == 40)
        out.append((st["passes"], st["events"], st["cg_iterations"], B.damage()[0], B.solution()))
        B.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    ctx.close()
