"""Which batches the library solves with the team CG: where it measured faster
than the launch path.  Few iterations: the choice is made before the first."""
import pytest

import amie_gpu as ag
import configs

pytestmark = pytest.mark.gpu


def cells3d(sizes):
    return [configs.rve3d(n, 9 + i) for i, n in enumerate(sizes)]


def cells(sizes):
    return [configs.rve(n, 7 + i, 0.3) for i, n in enumerate(sizes)]


# problems, precision, value-indexed, team (measured, time of the launches over the team's: 6.4, 1.7, 2.3, 0.75,
# 0.9, 1.3, 1.5, 0.75, 1.3)
CASES = {
    "patch": (lambda: [configs.config1(16)], ag.FP64, False, True),
    "cell": (lambda: cells([256]), ag.FP64, False, True),
    "small_cells": (lambda: cells([64] * 12), ag.FP64, False, True),
    "large_cells": (lambda: cells([384] * 4), ag.FP64, False, False),
    "mixed_sizes": (lambda: cells([512, 458, 404, 350, 296, 242, 188, 134]), ag.FP64, False, False),
    "large_cells_fix48": (lambda: cells([384] * 4), ag.MIXED_FIX48, False, True),
    "large_cells_indexed": (lambda: cells([384] * 4), ag.MIXED_FIX48, True, True),
    "cells_3d_indexed": (lambda: cells3d(range(19, 49, 3)), ag.MIXED_FIX48, True, False),
    "cells_3d": (lambda: cells3d([22, 26, 30, 34, 38, 42]), ag.MIXED_FIX48, False, True),
}


@pytest.mark.parametrize("case", list(CASES))
def test_choice(case):
    make, precision, indexed, team = CASES[case]
    ctx = ag.Context(0)
    B = ag.Batch(ctx, make())
    if indexed:
        B.set_spmv_kernel(precision, ag.JACOBI, 8, 8, 1)
    for _ in range(2):
        B.solve(precision=precision, maxit=5)
        assert B.team_info()["team_passes"] == (1 if team else 0)
    # asked for, it runs all the same
    B.set_team(ag.TEAM_ALWAYS)
    B.solve(precision=precision, maxit=5)
    assert B.team_info()["team_passes"] == 1
    B.set_team(ag.TEAM_NEVER)
    B.solve(precision=precision, maxit=5)
    assert B.team_info()["team_passes"] == 0
    B.close()
    ctx.close()
