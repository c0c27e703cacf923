"""The Gram's block skipping: state counts on either side of every 32-state block from 129 to 256
(the whole-chunk form) and around it (per tile pair), single plans against the FP64 oracle.  A
circuit of RY layers trimmed to the wanted parameter count.  Bar: the mixed path's 1e-6."""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


def _circuit(n, P):
    gates, k = [], 0
    while k < P:
        for q in range(n):
            for name in ("RY", "RZ"):
                p = k if k < P else -1
                gates.append((name, q, -1, p, 0.3 + 0.77 * k % 6.1))
                k += 1
        gates += [("CNOT", q, (q + 1) % n, -1, 0.0) for q in range(n)]
    return gates


@pytest.mark.parametrize("P", [1, 31, 32, 63, 95, 96, 127, 128, 159, 160, 191, 192, 223, 224, 255, 256, 287, 300])
def test_state_counts(P):
    n = 14
    ops, oops = Q.make_ops(_circuit(n, P)), O.make_ops(_circuit(n, P))
    p = Q.Plan(n, ops)
    got, st = p.execute()
    p.close()
    err = Q.rel_err(got, O.qgt(n, oops))
    print(f"P={P}: rel err {err:.2e}", flush=True)
    assert st["presplit"] == 1 and err <= 1e-6
