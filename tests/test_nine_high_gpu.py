"""Passes over nine high qubits with four contiguous low bits: the one-pass form at n = 22, and the
same group where the nine are not adjacent (n = 23 with one high qubit that carries no gate), against
the FP64 oracle on a block of rows from the first and columns from the last layers.

The states are FP32: per block of gates every amplitude gets about 2 roundings a qubit, unit norm, so an
inner product is off by at most about 4 n L 2^-24 (randomly signed, in practice its square root):
1e-6 against max |Q| = 1/4 is a quarter of that bound at n = 22.
"""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


def _ops(n, layers, bare):
    ops, p = [], 0
    for _ in range(layers):
        for t in ("RY", "RZ"):
            for q in range(n):
                if q != bare:
                    ops.append((t, q, -1, p, 0.1 + 0.37 * ((7 * p) % 17)))
                    p += 1
        ops += [("CNOT", q, (q + 1) % n, -1, 0.0) for q in range(n)]
    return ops, p


@pytest.mark.parametrize("n, bare", [(22, None), (23, 22), (23, 17)])
def test_nine_high_qubits(n, bare):
    lst, P = _ops(n, 2, bare)
    plan = Q.Plan(n, Q.make_ops(lst), Q.MODE_MIXED)
    Qm, _ = plan.execute()
    plan.close()
    rows = np.array([0, n - 3, P // 2 + 1], np.int32)
    cols = np.array([3, P // 2 - 2, P - n, P - 1], np.int32)
    ref = O.qgt_block(n, O.make_ops(lst), rows, cols)
    assert np.max(np.abs(Qm[np.ix_(rows, cols)] - ref)) <= 0.25e-6
    assert np.max(np.abs(Qm - Qm.conj().T)) <= 1e-12
