"""CNOT / SWAP / CZ stages folded into the passes (n > 13), into the resident kernel (4 <= n <= 13)
and the batched sweeps, and the stages that keep their per-gate kernels, against the FP64 oracle."""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu

TOL = 1e-6      # normwise; every element of a state takes ~2 FP32 roundings a gate: 60 x 2^-24 = 4e-6, randomly signed


def _stage(kind, n):
    if kind == "cz line":
        return [("CZ", q, q + 1) for q in range(n - 1)]
    if kind == "cnot line":
        return [("CNOT", q, q + 1) for q in range(n - 1)]
    if kind == "cz pairs":
        return [("CZ", a, b) for a in range(0, n, 3) for b in range(a + 1, n, 4)]
    if kind == "mixed":
        return [("CNOT", 0, n - 2), ("CZ", 0, n - 1), ("SWAP", 1, 2), ("CZ", 2, n - 2), ("CNOT", n - 1, 3), ("CZ", 3, 1),
                ("CNOT", 2, 0), ("CZ", 0, 1)] if n <= 13 else [
               ("CNOT", 11, n - 1), ("CZ", 0, n - 1), ("SWAP", 1, 2), ("CNOT", n - 1, 3), ("CZ", 3, 1), ("CNOT", 12, 13),
               ("CZ", 13, 5), ("CNOT", 3, 12), ("CZ", 12, 4)]
    if kind == "ring":
        return [("CNOT", q, (q + 1) % n) for q in range(n)]
    if kind == "apart":
        return [("SWAP", 1, n - 1), ("CZ", 0, n - 1), ("CNOT", 2, n - 1), ("CZ", 2, 3)]
    raise ValueError(kind)


def _circuit(n, kinds, bare=()):
    gates, k = [], 0
    for l, kind in enumerate(kinds):
        for t in ("RY", "RZ", "RX")[l % 2:][:2]:
            for q in range(n):
                if q in bare and l:
                    continue
                gates.append((t, q, -1, k, 0.2 + 0.61 * ((11 * k) % 13)))
                k += 1
        gates += [(t, a, b, -1, 0.0) for t, a, b in _stage(kind, n)]
    gates += [("RY", q, -1, k + q, 0.9 - 0.1 * q) for q in range(n)]
    return gates


@pytest.mark.parametrize("kinds", [("cz line", "cnot line", "cz line"), ("mixed", "cz pairs"), ("apart", "cz line", "mixed"),
                                   ("ring", "mixed", "ring"), ("cz line", "ring"), ("ring", "ring", "cz pairs")])
@pytest.mark.parametrize("n", [3, 4, 9, 13, 14, 15, 17])
def test_qgt(n, kinds):
    if n < 6 and "mixed" in kinds:
        kinds = tuple("cz line" if k == "mixed" else k for k in kinds)
    if n < 4:
        kinds = tuple("cnot line" if k == "apart" else k for k in kinds)
    gates = _circuit(n, kinds)
    ref = O.qgt(n, O.make_ops(gates))
    for opts in ({}, {"sweep_form": 1}, {"two_sided": False}, {"fused_inject": False}, {"presplit": False}):
        plan = Q.Plan(n, Q.make_ops(gates), Q.MODE_MIXED, **opts)
        for _ in range(3):      # eager, captured, replayed
            got, _ = plan.execute()
            assert Q.rel_err(got, ref) <= TOL, opts
        plan.close()


@pytest.mark.parametrize("n", [14, 16])
def test_layers_without_low_or_high_gates(n):
    """Blocks whose only pass is the one that carries the stage, and a qubit range without gates."""
    gates = _circuit(n, ("cz line", "mixed", "cz pairs"), bare=range(13))
    assert Q.rel_err(Q.qgt(n, Q.make_ops(gates)), O.qgt(n, O.make_ops(gates))) <= TOL
    for kinds in (("cz line", "mixed", "cz pairs"), ("cz line", "ring"), ("mixed", "cz pairs", "ring")):
        gates = _circuit(n, kinds, bare=range(13, n))
        assert Q.rel_err(Q.qgt(n, Q.make_ops(gates)), O.qgt(n, O.make_ops(gates))) <= TOL


@pytest.mark.parametrize("n", [3, 8, 13, 14])
def test_statevector_and_batch(n):
    kinds = ("cz line", "cnot line") if n < 6 else ("mixed", "cz line")
    gates = _circuit(n, kinds)
    psi = Q.statevector(n, Q.make_ops(gates))
    assert np.max(np.abs(psi - O.run(n, O.make_ops(gates)))) <= TOL
    if n <= 13:
        batch = Q.Batch([(n, Q.make_ops(gates)), (5, Q.make_ops(_circuit(5, ("cz line", "cz line"))))])
        out = batch.execute()[0]
        assert Q.rel_err(out[0], O.qgt(n, O.make_ops(gates))) <= TOL
        assert Q.rel_err(out[1], O.qgt(5, O.make_ops(_circuit(5, ("cz line", "cz line"))))) <= TOL
        batch.close()
    else:
        with pytest.raises(Q.QGTLError):
            Q.Batch([(n, Q.make_ops(gates))])


def _layers(n, kinds, seed):
    """One layer of random rotations and fixed gates per kind ("r" ring, "n" CNOT line, "z" CZ line)."""
    rng = np.random.default_rng(seed)
    gates, k = [], 0
    for kind in kinds:
        for q in range(n):
            if rng.integers(2):
                gates.append((str(rng.choice(["H", "S", "T", "SX", "X"])), q, -1, -1, 0.0))
            for _ in range(2):
                gates.append((str(rng.choice(["RX", "RY", "RZ"])), q, -1, k, rng.uniform(0.0, 2 * np.pi)))
                k += 1
        if kind == "r":
            gates += [("CNOT", q, (q + 1) % n, -1, 0.0) for q in range(n)]
        else:
            gates += [("CNOT" if kind == "n" else "CZ", q, q + 1, -1, 0.0) for q in range(n - 1)]
    return Q.make_ops(gates)


@pytest.mark.parametrize("n", [16, 17, 18])
@pytest.mark.parametrize("kinds", ["rnz", "rzz", "znr", "zzr", "nrz", "zrn", "nzn"])
def test_accuracy_of_rings_among_lines(n, kinds):
    """Circuits with a ring in some layer meet half way, on 22-bit Gram operands; those without one go to
    the end in complex64.  The rule looks at the gate list, not at how entangled the states are where
    they meet, so the accuracy is held here: the operands' rounding (2^-23) and the sweeps' (about 2^-24
    a gate on a qubit, seven gates, randomly signed: 1.6e-7) add to 2e-7 of an element of the largest size; a
    maximum over P^2 of them lies within twice that, of the mean over three circuits."""
    err = []
    for seed in range(3):
        ops = _layers(n, kinds, seed)
        ref = Q.qgt(n, ops, Q.MODE_FP64_PLAIN)
        err.append(Q.rel_err(Q.qgt(n, ops), ref))
    assert np.mean(err) <= 4e-7, err
