"""Team launches of several host threads: batches of their own contexts, the
same kernels with different amounts of LDS and numbers of workgroups."""
import threading

import numpy as np
import pytest

import amie_gpu as ag
from test_gpu_team import grids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ag.FP64, ag.MIXED_FIX48])
def test_threads(precision):
    sizes = [[15], [60], [90, 33], [150]]
    opts = dict(precision=precision, rtol=1e-10)

    def solve(n, times):
        ctx = ag.Context(0)
        out = []
        for _ in range(times):
            B = ag.Batch(ctx, grids(n))   # a plan of its own each time
            for _ in range(3):
                st = B.solve(**opts)
                assert st["status"] == 0
                info = B.team_info()
                assert info["team_passes"] == 1 and info["gave_up"] == 0, info
                out.append([B.solution(k).copy() for k in range(len(n))])
            B.close()
        ctx.close()
        return out

    alone = [solve(n, 1)[0] for n in sizes]
    got, failed = [None] * len(sizes), []

    def work(i):
        try:
            got[i] = solve(sizes[i], 4)
        except BaseException as e:
            failed.append((sizes[i], repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for ref, all_ in zip(alone, got):
        for xs in all_:
            for a, b in zip(xs, ref):
                np.testing.assert_array_equal(a, b)
