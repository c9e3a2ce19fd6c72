"""A server's step does not wait for the device: not for a group in flight
when another one's batch has been built."""
import time

import numpy as np
import pytest

import amie_gpu as ag
import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ag.FP64, ag.MIXED_FIX48])
def test_step_starts_a_group_without_waiting(precision):
    """Two cells of 448 and 440 cells a side, in two groups built at the same
    time, to rel. res 1e-12 (some 200 ms each): the second is started while
    the first is in flight, and no step takes as long as half of the first
    solve (a step that waits takes nearly all of it)."""
    big, small = configs.rve(448, 1, 0.3), configs.rve(440, 2, 0.3)
    ctx = ag.Context(0)
    B = ag.Batch(ctx, [big])
    B.solve(precision=precision, rtol=1e-12, maxit=8)
    t = time.perf_counter()
    st = B.solve(precision=precision, rtol=1e-12)
    alone = time.perf_counter() - t
    assert st["status"] == 0
    x = B.solution()
    B.close()
    S = ag.Server(ctx, 64 << 30, 8, precision=precision, rtol=1e-12)
    first = S.submit(big, 0., 0)
    while S.step(0.)[1]:   # queued until its batch is being built
        pass
    S.submit(small, 0., 0)
    steps, got, busy = [], {}, set()
    end = time.perf_counter() + 60
    while len(got) < 2 and time.perf_counter() < end:
        t = time.perf_counter()
        S.step(0.)
        steps.append(time.perf_counter() - t)
        for r in S.poll():
            got[r["ticket"]] = r["status"]
            busy.add(len(steps) - 1)   # it read a solution back
            if r["ticket"] == first:
                last = len(steps) - 1
                np.testing.assert_array_equal(S.solution(first, x.size), x.ravel())
    assert list(got.values()) == [0, 0]
    before = [s for k, s in enumerate(steps[:last]) if k not in busy]
    print("alone", alone, "longest step", max(before), flush=True)
    assert max(before) < 0.5 * alone
    S.close()
    ctx.close()
