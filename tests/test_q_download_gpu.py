"""Q written to the host by the finalizing kernel (up to 1 MB) or copied after it, in every order of
calls with and without Q: eager, captured without Q and replayed with it, and new angles between."""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, layers", [(2, 2), (6, 3), (14, 2), (14, 9), (15, 9)])   # P = 8, 36, 56, 252, 270: 270 is copied
def test_q_the_same_however_it_comes(n, layers):
    P = 2 * n * layers
    th = O.uniform_angles(3, P)
    ops = Q.hea_ops(n, layers, th)
    plan = Q.Plan(n, ops)
    first, _ = plan.execute()
    plan.close()
    assert np.array_equal(first, first.conj().T)
    for order in ((0, 0, 0, 1, 1), (1, 0, 1, 0, 1), (0, 1, 1, 0, 1)):
        plan = Q.Plan(n, ops)
        for want in order:
            out = np.full((P, P), np.nan + 0j) if want else None
            got, _ = plan.execute(want_q=bool(want), out=out)
            if want:
                assert np.array_equal(got, first)
        plan.set_angles(Q.hea_ops(n, layers, th[::-1].copy())["angle"])
        plan.execute(want_q=False)
        plan.set_angles(ops["angle"])
        assert np.array_equal(plan.execute()[0], first)
        plan.close()
