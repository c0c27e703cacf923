"""Small circuits whose states stay in LDS for the whole circuit (4 <= n <= 13, one launch):
every width the kernel is built for, against the FP64 oracle."""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-6


def _circuit(n, seed):
    """Gates with pre- and post-phases, qubits without a gate, CNOT / SWAP / CZ stages that are
    no ring, an empty stage and a trailing layer; 3 or more parameters per block."""
    rng = np.random.default_rng(seed)
    gates, k = [], 0

    def layer(names, skip):
        nonlocal k
        for q in range(n):
            if q == skip:
                continue
            name = names[rng.integers(len(names))]
            param = name in ("RX", "RY", "RZ")
            gates.append((name, q, -1, k if param else -1, float(rng.uniform(0, 2 * np.pi)) if param else 0.0))
            k += param

    for b in range(3):
        layer(["RX", "RY", "RZ"], b % n)
        layer(["H", "S", "T", "SX", "X", "RY"], (b + 2) % n)
        if b == 0:
            gates += [("CNOT", q, (q + 1) % n, -1, 0.0) for q in range(n)]
        elif b == 1:
            gates += [("SWAP", 0, n - 1, -1, 0.0), ("CNOT", n - 1, 1, -1, 0.0), ("CZ", 1, n - 2, -1, 0.0)]
    layer(["RX", "RZ"], -1)
    return gates


@pytest.mark.parametrize("n", [4, 5, 6, 7, 8, 9, 10, 11, 12, 13])
def test_resident_states_match_oracle(n):
    """Q, the overlaps' FP64 sums (through Q and energy_gradient) and a second execute at other
    angles.  Bar: the mixed path's 1e-6 normwise."""
    gates = _circuit(n, 60 + n)
    ops, oops = Q.make_ops(gates), O.make_ops(gates)
    p = Q.Plan(n, ops, Q.MODE_MIXED)
    p.set_hamiltonian(Q.tfim_terms(n, 1.0, 0.7))
    for turn in range(2):
        if turn:
            rng = np.random.default_rng(n)
            ang = np.where(ops["param"] >= 0, rng.uniform(0, 2 * np.pi, len(ops)), ops["angle"])
            p.set_angles(ang)
            oops["angle"] = ang
        got, st = p.execute()
        assert st["sweep_launches"] == 1
        e, g = p.energy_gradient()
        ref = O.qgt(n, oops)
        err = Q.rel_err(got, ref)
        print(f"n={n} P={p.P} turn {turn}: rel err {err:.2e}", flush=True)
        assert err <= MIXED_TOL
        e_ref, g_ref = O.tfim_gradient(n, oops, 1.0, 0.7)
        assert abs(e - e_ref) <= 1e-6 * max(1.0, abs(e_ref))
        assert np.max(np.abs(g - g_ref)) <= 1e-6 * max(1.0, np.max(np.abs(g_ref)))
    p.close()


@pytest.mark.parametrize("n,L", [(6, 1), (9, 3), (13, 1), (13, 10)])
def test_resident_rings_match_oracle(n, L):
    """The ansatz itself: one layer (every state injected in the last block) and more states
    than compute units (P = 260 at n = 13, L = 10)."""
    th = O.uniform_angles(900 + n, 2 * n * L)
    got = Q.qgt(n, Q.hea_ops(n, L, th))
    assert Q.rel_err(got, O.qgt(n, O.hea_ops(n, L, th))) <= MIXED_TOL
