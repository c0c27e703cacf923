"""The work whose speed counts: what a program that uses this library has it do, through the
library's Python view, at sizes from the smallest calls to the largest.

Kinds of case (the "kind" of a case):
  qgt      one quantum geometric tensor at new angles: Plan.set_angles + Plan.execute, Q in
           host memory.  The call of every loop that moves through parameter space; the
           circuit is the hardware-efficient ansatz (RY, RZ on each qubit, a CNOT ring).
  gates    the same call for a circuit of another shape: one random rotation and one fixed
           gate per qubit and layer, then CNOT or CZ along a line.
  batch    many independent circuits of uneven size in one call: Batch.set_angles +
           Batch.execute, the matrices in host memory (training sets, parameter scans).
  ng       one natural-gradient VQE step on a transverse-field Ising chain (angles -> QGT,
           energy, gradient -> Jacobi-PCG or Cholesky solve -> new angles).
  solve    (A + lambda I) x = b in FP64 for host matrices, one system or a batch.
  mlp      loss and gradient of one minibatch of the learned preconditioner's training.
  natgrad  the regularised natural gradient of QGTL's own C API (condition number, LU) for a
           complex Hermitian metric, as a program linked against QGTL's headers calls it.

The FP64 plain mode (one kernel per gate) is the fixed yardstick of the mixed path and no
case of its own.
"""
import ctypes
import math
import os
import random

import numpy as np
import torch

import quantum_geometric_tensor_amd as Q

_TUNE = os.path.join(os.path.dirname(os.path.abspath(Q.__file__)), "tune", "batch_hea_n12-18_L2-8.json")


def listed():
    return [
        # the smallest call: a few qubits, where launches and host work are all there is
        {"name": "qgt_n6_L3", "kind": "qgt", "n": 6, "L": 3},
        # the CPU-runnable configuration of the benchmark (P = 80)
        {"name": "qgt_n10_L4", "kind": "qgt", "n": 10, "L": 4},
        # an odd count, the largest state that one workgroup's tile holds (P = 156)
        {"name": "qgt_n13_L6", "kind": "qgt", "n": 13, "L": 6},
        # an ordinary odd size between the tile and the headline (P = 170)
        {"name": "qgt_n17_L5", "kind": "qgt", "n": 17, "L": 5},
        # the headline configuration (P = 240)
        {"name": "qgt_n20_L6", "kind": "qgt", "n": 20, "L": 6},
        # the largest single circuit that fits the card three times (P = 288, 37 GB of states)
        {"name": "qgt_n24_L6", "kind": "qgt", "n": 24, "L": 6},
        # a user's own ansatz: mixed gates and a line of entanglers instead of the ring
        {"name": "gates_n15_L4", "kind": "gates", "n": 15, "L": 4, "circuit": 1},
        # a parameter scan over uneven circuits (n 12..18, 2..8 layers), one batch
        {"name": "batch_128", "kind": "batch", "count": 128, "circuit": 0},
        # one step of the VQE loop at the learned preconditioner's size (P = 192)
        {"name": "ng_n16_L6", "kind": "ng", "n": 16, "L": 6, "method": "jacobi_pcg"},
        # the exact solve that produces training data and judges the iterative ones
        {"name": "solve_P192", "kind": "solve", "P": 192, "batch": 1, "method": "cholesky"},
        # one minibatch of the preconditioner's training (its defaults: width 256, rank 8, 256 samples)
        {"name": "mlp_P192_B256", "kind": "mlp", "P": 192, "rank": 8, "hidden": 256, "layers": 3, "B": 256},
        # the drop-in natural gradient for an ordinary metric
        {"name": "natgrad_P96", "kind": "natgrad", "P": 96},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["qgt"] * 6 + ["gates"] * 2 + ["batch", "ng", "solve", "mlp", "natgrad"])
    if kind == "qgt":
        return {"kind": "qgt", "n": rng.randint(4, 22), "L": rng.randint(2, 8)}
    if kind == "gates":
        return {"kind": "gates", "n": rng.randint(4, 18), "L": rng.randint(2, 6), "circuit": rng.randint(2, 10 ** 6)}
    if kind == "batch":
        return {"kind": "batch", "count": _log_int(rng, 4, 128), "circuit": rng.randint(1, 10 ** 6)}
    if kind == "ng":
        return {"kind": "ng", "n": rng.randint(6, 18), "L": rng.randint(2, 6),
                "method": rng.choice(["jacobi_pcg", "cholesky"])}
    if kind == "solve":
        P = _log_int(rng, 8, 512)
        return {"kind": "solve", "P": P, "batch": _log_int(rng, 1, max(1, (1 << 22) // (P * P)) if P > 256 else 64),
                "method": rng.choice(["cholesky", "jacobi_pcg"])}
    if kind == "mlp":
        return {"kind": "mlp", "P": rng.randint(32, 192), "rank": rng.choice([0, 4, 8, 16, 32]), "hidden": 256,
                "layers": 3, "B": _log_int(rng, 16, 512)}
    return {"kind": "natgrad", "P": _log_int(rng, 8, 192)}


# ---------------------------------------------------------------- inputs
_FIXED = ["H", "S", "T", "SX", "X"]
_ROT = ["RX", "RY", "RZ"]


def _line_circuit(n, L, circuit):
    """A circuit of random rotations and fixed gates with a line of CNOT or CZ after each layer."""
    g = random.Random(circuit)
    gates, k = [], 0
    for _ in range(L):
        for q in range(n):
            gates.append((g.choice(_FIXED), q, -1, -1, 0.0))
            gates.append((g.choice(_ROT), q, -1, k, 0.0))
            k += 1
            gates.append((g.choice(_ROT), q, -1, k, 0.0))
            k += 1
        two = g.choice(["CNOT", "CNOT", "CZ"])
        for q in range(n - 1):
            gates.append((two, q, q + 1, -1, 0.0))
    return gates, k


def _batch_shapes(case):
    g = random.Random(case["circuit"])
    return [(g.randint(12, 18), g.randint(2, 8)) for _ in range(case["count"])]


def _angles(seed, count):
    return np.random.default_rng([seed, count]).uniform(0.0, 2.0 * math.pi, count)


def _spd(P, rng, lo=1e-4):
    """A real metric-like matrix: eigenvalues from lo/4 to 1/4, random eigenvectors."""
    V, _ = np.linalg.qr(rng.standard_normal((P, P)))
    A = (V * (0.25 * np.logspace(math.log10(lo), 0, P))) @ V.T
    return 0.5 * (A + A.T)


def _solve_inputs(case, seed):
    rng = np.random.default_rng([seed, 1])
    P, batch = case["P"], case["batch"]
    A = np.stack([_spd(P, rng) for _ in range(batch)])
    b = rng.standard_normal((batch, P)) * 0.1
    return (A[0], b[0]) if batch == 1 else (A, b)


def _natgrad_inputs(case, seed):
    rng = np.random.default_rng([seed, 2])
    P = case["P"]
    V, _ = np.linalg.qr(rng.standard_normal((P, P)) + 1j * rng.standard_normal((P, P)))
    M = (V * (0.25 * np.logspace(-4, 0, P))) @ V.conj().T
    M = (0.5 * (M + M.conj().T)).astype(np.complex64)
    M = np.tril(M, -1) + np.tril(M, -1).conj().T + np.diag(M.diagonal().real)
    g = (rng.standard_normal(P) * 0.1).astype(np.complex64)
    return np.ascontiguousarray(M, np.complex64), g


def _mlp_inputs(case, seed):
    """Weights, features and Jacobi-scaled metrics of a training set of twice the minibatch."""
    rng = np.random.default_rng([seed, 3])
    P, B = case["P"], case["B"]
    S = 2 * B
    gen = torch.Generator().manual_seed(seed)
    F = torch.randn((S, P, P // 2), generator=gen, dtype=torch.float32)
    A = torch.bmm(F, F.transpose(1, 2).contiguous()) / (P // 2) * 0.2 + 0.05 * torch.eye(P)
    D = torch.diagonal(A, dim1=1, dim2=2)
    s = 1.0 / torch.sqrt(D)
    As = (A * s[:, :, None] * s[:, None, :]).numpy()
    theta = rng.uniform(0, 2 * math.pi, (S, P))
    X = np.concatenate([np.sin(theta), np.cos(theta), np.log(D.numpy()), rng.uniform(0.5, 1.5, (S, 1))],
                       1).astype(np.float32)
    dims = _mlp_dims(case)
    w = []
    for i, (a, b) in enumerate(dims):
        lim = math.sqrt(3.0 / a) * (0.2 if i == len(dims) - 1 else 1.0)
        w.append(rng.uniform(-lim, lim, a * b).astype(np.float32))
        w.append((0.01 * rng.standard_normal(b)).astype(np.float32))
    idx = rng.permutation(S)[:B].astype(np.int32)
    return np.concatenate(w), X, As, idx


def _mlp_dims(case):
    P, H = case["P"], case["hidden"]
    widths = [3 * P + 1] + [H] * case["layers"] + [P * (1 + case["rank"])]
    return list(zip(widths[:-1], widths[1:]))


class _NGConfig(ctypes.Structure):
    """natural_gradient_config_t of QGTL's quantum_geometric_gradient.h."""
    _fields_ = [("regularization_param", ctypes.c_float), ("condition_threshold", ctypes.c_float),
                ("use_adaptive_regularization", ctypes.c_bool), ("use_pseudoinverse_fallback", ctypes.c_bool),
                ("singular_value_cutoff", ctypes.c_float)]


def _natgrad_function():
    f = Q.lib().compute_regularized_natural_gradient
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.POINTER(_NGConfig)]
    f.restype = ctypes.c_bool
    return f


_METHOD = {"cholesky": Q.SOLVE_CHOLESKY, "jacobi_pcg": Q.SOLVE_JACOBI_PCG}
_NG = {"lam": 1e-3, "eta": 0.1, "tol": 1e-8}


def _circuit(case, seed):
    """(n, ops) at the seed's angles."""
    n = case["n"]
    if case["kind"] == "gates":
        gates, P = _line_circuit(n, case["L"], case["circuit"])
        th = _angles(seed, P)
        return n, Q.make_ops([(g, a, b, k, th[k] if k >= 0 else 0.0) for g, a, b, k, _ in gates])
    return n, Q.hea_ops(n, case["L"], _angles(seed, 2 * n * case["L"]))


def _field(seed):
    return 0.5 + random.Random(seed).random()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("qgt", "gates"):
        n, ops = _circuit(case, seed)
        plan = Q.Plan(n, ops)
        return {"kind": kind, "plan": plan, "angles": ops["angle"].copy(), "Q": np.empty((plan.P, plan.P), np.complex128)}
    if kind == "batch":
        circuits = []
        for i, (n, L) in enumerate(_batch_shapes(case)):
            circuits.append((n, Q.hea_ops(n, L, _angles(seed * 1000 + i, 2 * n * L))))
        b = Q.Batch(circuits, Q.load_batch_tune(_TUNE))
        return {"kind": kind, "batch": b, "angles": [ops["angle"].copy() for _, ops in circuits],
                "Q": np.empty(b.q_size, np.complex128)}
    if kind == "ng":
        n, ops = _circuit(case, seed)
        plan = Q.Plan(n, ops)
        plan.set_hamiltonian(Q.tfim_terms(n, 1.0, _field(seed)))
        return {"kind": kind, "plan": plan, "theta": _angles(seed, 2 * n * case["L"]), "method": _METHOD[case["method"]]}
    if kind == "solve":
        A, b = _solve_inputs(case, seed)
        return {"kind": kind, "A": A, "b": b, "method": _METHOD[case["method"]]}
    if kind == "mlp":
        w, X, As, idx = _mlp_inputs(case, seed)
        m = Q.MLP(X.shape[1], case["hidden"], case["layers"], case["P"], case["rank"])
        m.set_params(w)
        m.set_data(X, As)
        return {"kind": kind, "mlp": m, "idx": idx}
    M, g = _natgrad_inputs(case, seed)
    return {"kind": kind, "M": M, "g": g, "x": np.empty_like(g), "f": _natgrad_function(),
            "config": _NGConfig(1e-4, 1e8, True, True, 1e-10)}


def run(state):
    kind = state["kind"]
    if kind in ("qgt", "gates"):
        state["plan"].set_angles(state["angles"])
        state["plan"].execute(out=state["Q"])
        return state["Q"]
    if kind == "batch":
        state["batch"].set_angles(state["angles"])
        state["batch"].execute(out=state["Q"])
        return state["Q"]
    if kind == "ng":
        theta = state["theta"].copy()
        info = Q.ng_step(state["plan"], theta, _NG["lam"], _NG["eta"], state["method"], _NG["tol"], 20000)
        return {"theta": theta, "energy": info["energy"], "grad_norm": info["grad_norm"],
                "step_norm": info["step_norm"]}
    if kind == "solve":
        x, _ = Q.solve(state["A"], state["b"], 1e-3, state["method"], tol=1e-10)
        return x
    if kind == "mlp":
        loss, grad = state["mlp"].loss_grad(state["idx"])
        return {"loss": loss, "grad": grad}
    x = state["x"]
    if not state["f"](state["g"].ctypes.data, state["M"].ctypes.data, x.ctypes.data, x.size,
                      ctypes.byref(state["config"])):
        raise RuntimeError("compute_regularized_natural_gradient failed")
    return x


# ---------------------------------------------------------------- work
def _qgt_work(n, P, ngates):
    """Bytes: the angles in, Q out.  Operations: the Hermitian half of the complex Gram, and one
    2 x 2 complex product per gate on the state itself (the derivative states could be carried
    by fewer passes than any present schedule's, so they are left out)."""
    N = 1 << n
    return {"bytes": 8.0 * ngates + 16.0 * P * P, "flops": 4.0 * N * P * (P + 1) + 14.0 * N * ngates}


def work(case):
    kind = case["kind"]
    if kind == "qgt":
        return _qgt_work(case["n"], 2 * case["n"] * case["L"], 2 * case["n"] * case["L"])
    if kind == "gates":
        return _qgt_work(case["n"], 2 * case["n"] * case["L"], 3 * case["n"] * case["L"])
    if kind == "batch":
        parts = [_qgt_work(n, 2 * n * L, 2 * n * L) for n, L in _batch_shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "ng":
        P = 2 * case["n"] * case["L"]
        w = _qgt_work(case["n"], P, P)
        return {"bytes": 16.0 * P, "flops": w["flops"] + P ** 3 / 3.0 + 8.0 * P * 2 ** case["n"]}
    if kind == "solve":
        P, batch = case["P"], case["batch"]
        return {"bytes": batch * 8.0 * (P * P + 2 * P), "flops": batch * P ** 3 / 3.0}
    if kind == "mlp":
        P, r, B = case["P"], case["rank"], case["B"]
        weights = sum(a * b for a, b in _mlp_dims(case))
        params = weights + sum(b for _, b in _mlp_dims(case))
        return {"bytes": 4.0 * B * (P * P + 3 * P + 1) + 8.0 * params,
                "flops": 6.0 * B * weights + 2.0 * B * P * P * r}
    P = case["P"]
    return {"bytes": 8.0 * (P * P + 2 * P), "flops": 8.0 * P ** 3 / 3.0}


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    """About four times the largest distance from the FP64 result measured over the listed and
    some drawn cases."""
    kind = case["kind"]
    if kind in ("qgt", "gates", "batch"):
        # complex64 sweeps, 22-bit Gram operands, fp32 sums: 2.6e-7 and (an off-diagonal element
        # near zero against the root mean square) 1.0e-5 measured
        return {"rel": 1e-6, "max": 4e-5}
    if kind == "ng":
        # a rounding of Q is divided by the shift in x = (Re Q + 1e-3 I)^-1 grad E: 3.6e-6 measured
        # (the step's norm; the new angles themselves 1e-7)
        return {"rel": 1.5e-5}
    if kind == "solve":
        # FP64 throughout: 7e-15 measured; the iterative method stops at a residual of 1e-10 and
        # the shifted matrix has a condition number of about 250
        return {"rel": 1e-13} if case["method"] == "cholesky" else {"rel": 1e-7}
    if kind == "mlp":
        # bf16 operands of the dense layers: 3.5e-3 measured (the gradient)
        return {"rel": 1.4e-2}
    # QGTL's ComplexFloat result: 2.8e-8 measured
    return {"rel": 1.2e-7}


# ---------------------------------------------------------------- FP64 results
_S2 = 1.0 / math.sqrt(2.0)
_FIXED_M = {"H": [[_S2, _S2], [_S2, -_S2]], "S": [[1, 0], [0, 1j]], "T": [[1, 0], [0, complex(_S2, _S2)]],
            "SX": [[0.5 + 0.5j, 0.5 - 0.5j], [0.5 - 0.5j, 0.5 + 0.5j]], "X": [[0, 1], [1, 0]],
            "Z": [[1, 0], [0, -1]]}
_GEN = {"RX": [[0, 1], [1, 0]], "RY": [[0, -1j], [1j, 0]], "RZ": [[1, 0], [0, -1]]}


def _rot(name, t):
    return math.cos(t / 2) * np.eye(2) - 1j * math.sin(t / 2) * np.array(_GEN[name], complex)


class _States:
    """Rows of complex128 states: row 0 the state, row 1 + k the derivative by parameter k."""

    def __init__(self, n, P):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.n, self.rows = n, 1
        self.D = torch.zeros((1 + P, 1 << n), dtype=torch.complex128, device=dev)
        self.D[0, 0] = 1.0

    def _pairs(self, rows, q):
        return self.D[rows].view(-1, 1 << (self.n - 1 - q), 2, 1 << q)

    def one(self, m, q, rows=None):
        m = np.asarray(m, complex)
        rows = slice(0, self.rows) if rows is None else rows
        step = max(1, (1 << 26) >> self.n)
        for r in range(rows.start, rows.stop, step):
            v = self._pairs(slice(r, min(rows.stop, r + step)), q)
            a, b = v[:, :, 0].clone(), v[:, :, 1].clone()
            v[:, :, 0] = complex(m[0, 0]) * a + complex(m[0, 1]) * b
            v[:, :, 1] = complex(m[1, 0]) * a + complex(m[1, 1]) * b

    def derive(self, name, q):
        self.D[self.rows] = self.D[0]
        self.one(-0.5j * np.array(_GEN[name], complex), q, slice(self.rows, self.rows + 1))
        self.rows += 1

    def permute(self, pairs):
        """CNOT(c -> t) for (c, t) in order."""
        x = torch.arange(1 << self.n, device=self.D.device)
        src = x
        for c, t in reversed(pairs):          # the source of y: undo the gates from the last
            src = src ^ (((src >> c) & 1) << t)
        step = max(1, (1 << 26) >> self.n)
        for r in range(0, self.rows, step):
            s = slice(r, min(self.rows, r + step))
            self.D[s] = self.D[s].index_select(1, src)

    def cz(self, c, t):
        x = torch.arange(1 << self.n, device=self.D.device)
        self.D[:self.rows] *= 1.0 - 2.0 * (((x >> c) & (x >> t)) & 1).to(torch.float64)


def _evolve(n, layers, P):
    """layers: lists of ("one", name, q, angle, is_param) / ("cnots", pairs) / ("cz", c, t)."""
    st = _States(n, P)
    for op in layers:
        if op[0] == "one":
            _, name, q, angle, is_param = op
            st.one(_rot(name, angle) if name in _GEN else _FIXED_M[name], q)
            if is_param:
                st.derive(name, q)
        elif op[0] == "cnots":
            st.permute(op[1])
        else:
            st.cz(op[1], op[2])
    return st


def _hea_layers(n, L, th):
    out = []
    for l in range(L):
        out += [("one", "RY", q, th[2 * n * l + q], True) for q in range(n)]
        out += [("one", "RZ", q, th[2 * n * l + n + q], True) for q in range(n)]
        out.append(("cnots", [(q, (q + 1) % n) for q in range(n)]))
    return out


def _line_layers(case, th):
    gates, _ = _line_circuit(case["n"], case["L"], case["circuit"])
    out = []
    for name, a, b, k, _ in gates:
        if name == "CZ":
            out.append(("cz", a, b))
        elif name == "CNOT":
            if out and out[-1][0] == "cnots":
                out[-1][1].append((a, b))
            else:
                out.append(("cnots", [(a, b)]))
        else:
            out.append(("one", name, a, th[k] if k >= 0 else 0.0, k >= 0))
    return out


def _qgt_of(st):
    D, psi = st.D[1:], st.D[0]
    G = torch.zeros((D.shape[0], D.shape[0]), dtype=torch.complex128, device=D.device)
    a = torch.zeros(D.shape[0], dtype=torch.complex128, device=D.device)
    step = 1 << 18
    for k in range(0, D.shape[1], step):
        d = D[:, k:k + step].contiguous()
        G += d.conj().resolve_conj() @ d.T.contiguous()
        a += d.conj().resolve_conj() @ psi[k:k + step].contiguous()
    return (G - a[:, None] * a.conj()[None, :]).cpu().numpy()


def _refined_solve(A, b):
    """A x = b with residuals in extended precision."""
    x = np.linalg.solve(A, b).astype(np.longdouble)
    Al, bl = A.astype(np.longdouble), b.astype(np.longdouble)
    for _ in range(3):
        r = bl - (Al * x[None, :]).sum(1)
        x = x + np.linalg.solve(A, r.astype(np.float64))
    return x.astype(np.float64)


def _exact_qgt(n, layers, P):
    return _qgt_of(_evolve(n, layers, P))


def _exact_ng(case, seed):
    n, L = case["n"], case["L"]
    P = 2 * n * L
    th = _angles(seed, P)
    st = _evolve(n, _hea_layers(n, L, th), P)
    psi = st.D[0]
    x = torch.arange(1 << n, device=psi.device)
    z = [1.0 - 2.0 * ((x >> q) & 1).to(torch.float64) for q in range(n)]
    diag = torch.zeros(1 << n, dtype=torch.float64, device=psi.device)
    for q in range(n - 1):
        diag -= z[q] * z[q + 1]
    hpsi = diag * psi
    h = _field(seed)
    for q in range(n):
        hpsi = hpsi - h * psi[x ^ (1 << q)]
    E = float((psi.conj() * hpsi).sum().real)
    g = 2.0 * (st.D[1:].conj().resolve_conj() @ hpsi).real.cpu().numpy()
    A = _qgt_of(st).real + _NG["lam"] * np.eye(P)
    step = _NG["eta"] * _refined_solve(A, g)
    return {"theta": th - step, "energy": E, "grad_norm": float(np.linalg.norm(g)),
            "step_norm": float(np.linalg.norm(step))}


def _exact_mlp(case, seed):
    w, X, As, idx = _mlp_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    P, r, B = case["P"], case["rank"], case["B"]
    p = torch.tensor(w, dtype=torch.float64, device=dev, requires_grad=True)
    h = torch.tensor(X[idx], dtype=torch.float64, device=dev)
    o, dims = 0, _mlp_dims(case)
    for i, (a, b) in enumerate(dims):
        z = h @ p[o:o + a * b].view(a, b) + p[o + a * b:o + a * b + b]
        o += a * b + b
        h = torch.nn.functional.gelu(z, approximate="tanh") if i < len(dims) - 1 else z
    y = h.view(B, P, 1 + r)
    s, u = y[:, :, 0], y[:, :, 1:] / math.sqrt(P)
    total = 0.0
    for k in range(B):
        A = torch.tensor(As[idx[k]], dtype=torch.float64, device=dev)
        tr = (torch.exp(s[k]) * torch.diagonal(A)).sum() + (u[k] * (A @ u[k])).sum()
        W = torch.eye(r, dtype=torch.float64, device=dev) + u[k].T.contiguous() @ (torch.exp(-s[k])[:, None] * u[k])
        logdet = torch.logdet(W) if r > 0 else 0.0
        total = total + P * torch.log(tr / P) - s[k].sum() - logdet
    loss = total / B
    loss.backward()
    return {"loss": float(loss.detach()), "grad": p.grad.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qgt", "gates"):
        n, L = case["n"], case["L"]
        P = 2 * n * L
        if (P + 1) << n > 1 << 29:
            return None                       # 8 GB and more of complex128 states
        th = _angles(seed, P)
        return _exact_qgt(n, _hea_layers(n, L, th) if kind == "qgt" else _line_layers(case, th), P)
    if kind == "batch":
        if case["count"] > 160:
            return None
        out = []
        for i, (n, L) in enumerate(_batch_shapes(case)):
            P = 2 * n * L
            out.append(_exact_qgt(n, _hea_layers(n, L, _angles(seed * 1000 + i, P)), P).reshape(-1))
        return np.concatenate(out)
    if kind == "ng":
        return _exact_ng(case, seed)
    if kind == "solve":
        A, b = _solve_inputs(case, seed)
        shift = 1e-3 * np.eye(case["P"])
        if case["batch"] == 1:
            return _refined_solve(A + shift, b)
        return np.stack([_refined_solve(A[i] + shift, b[i]) for i in range(case["batch"])])
    if kind == "mlp":
        return _exact_mlp(case, seed)
    M, g = _natgrad_inputs(case, seed)
    x = np.linalg.solve(M.astype(np.complex128) + float(np.float32(1e-4)) * np.eye(case["P"]), g.astype(np.complex128))
    return x
