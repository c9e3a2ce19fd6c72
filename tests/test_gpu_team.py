"""The team CG (a problem's rows held by a few resident workgroups for a whole
pass) against the launch path, which time_kernels keeps: the same sums in the
same order, so solutions, iterations, refinements and statuses are equal bit
for bit and no tolerance is involved.
"""
import numpy as np
import pytest

import amie_gpu as ag
import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ag.Context(0)
    yield c
    c.close()


def remade(p, **kw):
    """The problem with other arrays."""
    args = dict(phase=p.phase, damage=p.damage, bc_dofs=p.bc_dofs, bc_vals=p.bc_vals)
    cmats = kw.pop("cmats", p.cmats)
    return ag.Problem(p.etype, p.coords, p.conn, cmats, **{**args, **kw})


def grids(sizes, seed=5):
    """Two-phase P1 squares: one to many tiles, the last one part filled."""
    rng = np.random.default_rng(seed)
    probs = [configs.config1(n) for n in sizes]
    return [remade(p, cmats=configs.composite_cmats(), phase=rng.integers(0, 2, size=p.conn.shape[0])) for p in probs]


def with_nan(p):
    return remade(p, bc_vals=np.concatenate([p.bc_vals[:-1], [np.nan]]))


def homogeneous(p):
    return remade(p, bc_vals=np.zeros_like(p.bc_vals))


# (256 rows a tile; one member keeps at most four; sums of more than 64 tiles
# take two hops)
CASES = {
    "one_tile_and_ragged": lambda: grids([1, 7, 15, 16, 22]),
    "four_and_five_tiles": lambda: grids([30, 31, 32, 35]),
    "64_and_65_tiles": lambda: grids([126, 127, 128]),
    "many_tiles": lambda: grids([290, 20]),
    "p2": lambda: [configs.config2(n, seed=9) for n in (3, 21, 70)],
    "tet4": lambda: [configs.config3(n, seed=8) for n in (2, 9, 26)],
    "rve_three_loads": lambda: [configs.rve(n, 40 + n, 0.3) for n in (5, 31, 33, 130)],
    "rve3d_three_loads": lambda: [configs.rve3d(n, 3, macro=1e-3 * np.eye(6)[:3]) for n in (3, 12)],
    "homogeneous_and_not": lambda: [homogeneous(configs.config1(20)), configs.config1(40)],
    "nan": lambda: [with_nan(configs.config1(20)), configs.config1(40)],
}


@pytest.mark.parametrize("matrix", ["fp64", "fix48", "indexed"])
@pytest.mark.parametrize("precond", [ag.JACOBI, ag.BLOCK_JACOBI])
@pytest.mark.parametrize("case", list(CASES))
def test_team_solve_matches_launches(ctx, case, precond, matrix):
    probs = CASES[case]()
    prec = ag.FP64 if matrix == "fp64" else ag.MIXED_FIX48
    if matrix == "indexed" and case == "tet4":   # blocks that repeat: no damage, coordinates without rounding
        probs = [remade(configs.config3(n), damage=None) for n in (2, 8, 16)]
    B = ag.Batch(ctx, probs)
    if matrix == "indexed":
        B.set_spmv_kernel(prec, precond, 8, 8, 1)
    for kw in (dict(rtol=1e-10), dict(rtol=1e-10, stall_iters=16, ckpt_interval=8), dict(rtol=1e-12, maxit=37)):
        print(case, precond, matrix, kw, flush=True)
        ref = B.solve(precision=prec, precond=precond, time_kernels=1, **kw)
        xr = [B.solution(k).copy() for k in range(len(probs))]
        ir = [B.problem_info(k) for k in range(len(probs))]
        for again in range(2):   # the second pass finds the first one's exchange words
            got = B.solve(precision=prec, precond=precond, **kw)
            for k in range(len(probs)):
                np.testing.assert_array_equal(B.solution(k), xr[k])
                assert repr(B.problem_info(k)) == repr(ir[k]), (k, again)
            for key in ("status", "iterations_max", "iterations_sum", "refinements", "nproblems_converged",
                        "nproblems_escalated"):
                assert got[key] == ref[key], (key, again)
    B.close()
