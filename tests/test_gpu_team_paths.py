"""The team CG at every number of slices a wavefront holds, and its sums over
more tiles than one trip of their loop takes, against the launch path: the
same sums in the same order, so the results are equal bit for bit and no
tolerance is involved.  team_info says how a solve ran, so that no case
compares the launch path with itself.
"""
import numpy as np
import pytest

import amie_gpu as ag
import configs
from test_gpu_team import grids, remade

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ag.Context(0)
    yield c
    c.close()


def rves3d():
    return [configs.rve3d(n, 3, macro=1e-3 * np.eye(6)[:3]) for n in (14, 4)]


# problems of several members at the most tiles a workgroup takes (of 256
# rows), and one or two of a single member with a part-filled tile
CASES = {
    "p1": lambda: grids([150, 63, 22]),
    "p2": lambda: [configs.config2(n, seed=9) for n in (75, 17)],
    "rve": lambda: [configs.rve(n, 40 + n, 0.3) for n in (130, 47, 9)],
    "tet4": lambda: [configs.config3(n, seed=8) for n in (26, 13)],
    "rve3d": rves3d,
}
# most tiles of a workgroup: a slice's y, r and q take 6 (FP64) or 4 (FP32
# vectors) registers a DOF and right-hand side, at most 96 in 1, 2, 4 or 8
# slices a wavefront; 8 wavefronts, 4 slices a tile
MOST = {("fp64", "p1"): 16, ("fp64", "p2"): 16, ("fp64", "rve"): 4, ("fp64", "tet4"): 8, ("fp64", "rve3d"): 2,
        ("fp32", "p1"): 16, ("fp32", "p2"): 16, ("fp32", "rve"): 8, ("fp32", "tet4"): 16, ("fp32", "rve3d"): 4}


def compare(B, n, prec, precond, tiles, tiles64, **kw):
    """tiles64: of a second pass, the stalled problems' in FP64."""
    ref = B.solve(precision=prec, precond=precond, time_kernels=1, **kw)
    assert B.team_info()["team_passes"] == 0
    xr = [B.solution(k).copy() for k in range(n)]
    ir = [repr(B.problem_info(k)) for k in range(n)]
    for again in range(2):
        got = B.solve(precision=prec, precond=precond, **kw)
        info = B.team_info()
        assert info["team_passes"] == info["passes"] > 0, info
        assert info["tiles"] == (tiles if info["passes"] == 1 else tiles64), info
        for k in range(n):
            np.testing.assert_array_equal(B.solution(k), xr[k])
            assert repr(B.problem_info(k)) == ir[k], (k, again)
        for key in ("status", "iterations_max", "iterations_sum", "refinements", "nproblems_converged",
                    "nproblems_escalated"):
            assert got[key] == ref[key], (key, again)


@pytest.mark.parametrize("matrix", ["fp64", "fix48", "indexed"])
@pytest.mark.parametrize("precond", [ag.JACOBI, ag.BLOCK_JACOBI])
@pytest.mark.parametrize("case", list(CASES))
def test_every_slice_count_matches_launches(ctx, case, precond, matrix):
    """1, 2, 3, 4, 8 and 16 tiles a workgroup (3: the last slices of a
    wavefront's share are absent), which are 1, 2, 4 and 8 slices a
    wavefront."""
    probs = CASES[case]()
    prec = ag.FP64 if matrix == "fp64" else ag.MIXED_FIX48
    if matrix == "indexed" and case == "tet4":   # blocks that repeat: no damage, coordinates without rounding
        probs = [remade(configs.config3(n), damage=None) for n in (16, 8)]
    B = ag.Batch(ctx, probs)
    if matrix == "indexed":
        B.set_spmv_kernel(prec, precond, 8, 8, 1)
    most, most64 = MOST["fp64" if matrix == "fp64" else "fp32", case], MOST["fp64", case]
    for tiles in [t for t in (1, 2, 3, 4, 8, 16) if t <= most]:
        B.set_team(ag.TEAM_ALWAYS, tiles)
        print(case, precond, matrix, tiles, flush=True)
        compare(B, len(probs), prec, precond, tiles, min(tiles, most64), rtol=1e-9, stall_iters=16, ckpt_interval=8)
    compare(B, len(probs), prec, precond, most, most64, rtol=1e-12, maxit=37)
    B.close()


@pytest.mark.parametrize("matrix", ["fp64", "fix48", "indexed"])
def test_sums_over_more_tiles_than_a_trip(ctx, matrix):
    """2 061 tiles (the sums of a value take 8 x 256 tiles a trip), over the
    few iterations that an unconverged solve of 37 makes."""
    probs = grids([725])
    B = ag.Batch(ctx, probs)
    prec = ag.FP64 if matrix == "fp64" else ag.MIXED_FIX48
    if matrix == "indexed":
        B.set_spmv_kernel(prec, ag.JACOBI, 8, 8, 1)
    B.set_team(ag.TEAM_ALWAYS)
    B.solve(precision=prec, maxit=5)
    tiles = B.team_info()["tiles"]
    assert tiles >= 8, tiles
    compare(B, 1, prec, ag.JACOBI, tiles, tiles, rtol=1e-12, maxit=37)
    B.close()


def test_team_choice(ctx):
    probs = grids([40])
    B = ag.Batch(ctx, probs)
    B.set_team(ag.TEAM_NEVER)
    B.solve(precision=ag.FP64)
    info = B.team_info()
    assert info["passes"] == 1 and not any(v for k, v in info.items() if k != "passes")
    B.set_team(ag.TEAM_ALWAYS, 2)
    B.solve(precision=ag.FP64)
    info = B.team_info()
    assert info["halo_rows"] > 0
    assert info == dict(info, passes=1, team_passes=1, tiles=2, workgroups=4)   # 1 681 rows, 7 tiles
    B.solve(precision=ag.MIXED)   # no team kernel for this precision
    assert B.team_info()["team_passes"] == 0
    for bad in ((4, 0), (-1, 0), (0, -1)):
        with pytest.raises(ag.AmieError):
            B.set_team(*bad)
    B.close()
