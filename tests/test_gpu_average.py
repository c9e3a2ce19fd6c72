"""Average stresses: sums over chunks of 1 024 elements, then over the chunks."""
import numpy as np
import pytest

import amie_gpu as ag
import configs
import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("etype,sizes", [("p1", (1, 22, 23, 32, 33)), ("p2", (2, 23, 32)), ("tet4", (2, 5, 6, 8))])
def test_average_stress_over_chunks(etype, sizes):
    """Element counts below, at and above one and two chunks in one batch
    (P1, P2: 2 n^2; Tet4: 6 n^3), against the volume average of the strains
    of the device's displacements.  Each of the at most 3 072 terms of a sum
    carries a few roundings: 3 072 * 4 * 2^-53 < 2e-12 of the largest term's
    size bounds both sides together."""
    make = {"p1": lambda n: configs.rve(n, 60 + n, 0.3), "p2": lambda n: configs.config2(n, seed=n),
            "tet4": lambda n: configs.config3(n, seed=n)}[etype]
    ctx = ag.Context(0)
    probs = [make(n) for n in sizes]
    B = ag.Batch(ctx, probs)
    st = B.solve(precision=ag.FP64, rtol=1e-10)
    assert st["status"] == 0, st
    got = B.average_stress()
    for p, prob in enumerate(probs):
        for k in range(B.nrhs):
            eps = B.element_strain(p, k)
            if prob.damage is not None:   # C (1 - d) eps
                eps = eps * (1. - prob.damage)[:, None]
            ref, _ = orc.average_stress(prob.etype, prob.conn, prob.coords, prob.cmats, prob.phase, eps)
            stress = np.abs(prob.cmats).max() * np.abs(eps).max()
            np.testing.assert_allclose(got[p][k], ref, rtol=0, atol=2e-12 * stress)
    B.close()
    ctx.close()
