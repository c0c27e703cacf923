"""Dense layers of the preconditioner's network at the edges of the products' tiles: widths that
are no multiple of the 32 x 32 tile or of the vector loads, K past one 256-wide stage, batches
below and above a tile, rank 0 -- against the FP64 oracle given the same bf16-rounded weights and
inputs.  Bars: the bf16 ones of tests/test_mlp_gpu.py (forward 6e-3, loss 1e-2, gradient 1e-2
normwise, cosine 0.9999)."""
import numpy as np
import pytest

import oracle_lib as O
import quantum_geometric_tensor_amd as Q
from test_mlp_gpu import bf16, oracle_params, spd_unit_diag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,H,nh,P,r,B", [(301, 33, 1, 7, 3, 70), (22, 260, 2, 9, 0, 5), (64, 64, 3, 33, 8, 257),
                                          (577, 256, 3, 12, 4, 33), (5, 300, 1, 65, 15, 64)])
def test_layers_match_oracle(F, H, nh, P, r, B):
    m = Q.MLP(F, H, nh, P, r, seed=F + H)
    p = m.get_params()
    p *= 3.0                                     # a non-trivial output from the small initial output layer
    m.set_params(p)
    rng = np.random.default_rng(B)
    S = B + 3
    X = rng.normal(size=(S, F)).astype(np.float32)
    As = np.stack([spd_unit_diag(P, 10 + s % 7) for s in range(S)]).astype(np.float32)
    Y = m.forward(X[:B]).astype(np.float64)
    Yo = O.mlp_forward(F, H, nh, m.out_dim, oracle_params(m), bf16(X[:B]))
    assert np.max(np.abs(Y - Yo)) <= 6e-3 * np.max(np.abs(Yo))
    m.set_data(X, As)
    idx = rng.permutation(S)[:B].astype(np.int32)
    loss, g = m.loss_grad(idx)
    lo, go = O.mlp_loss_grad(F, H, nh, P, r, oracle_params(m), bf16(X[idx]), As[idx].astype(np.float64))
    cos = float(np.dot(g, go) / (np.linalg.norm(g) * np.linalg.norm(go)))
    print(f"loss {loss:.6f} oracle {lo:.6f} grad err {np.max(np.abs(g - go)) / np.max(np.abs(go)):.2e} cos {cos:.6f}")
    assert abs(loss - lo) <= 1e-2 * max(1.0, abs(lo))
    assert np.max(np.abs(g - go)) <= 1e-2 * np.max(np.abs(go)) and cos >= 0.9999
    m.close()


@pytest.mark.parametrize("P,r", [(3, 1), (17, 16), (31, 17), (200, 10), (255, 32), (481, 17), (1023, 8)])
def test_loss_kernel_sizes(P, r):
    """(P = 1 is left out: its loss is zero whatever y is.)  The loss kernel's forms (rank up to 16 and up to 32, both LDS sizes, odd P without vector
    loads).  A network of one narrow layer, so the gradient of the output bias is the kernel's
    own dL/dy summed over the samples.  Loss: FP64 but for the network's bf16 output error (bar as
    above); the output bias' gradient: 3.5e-2 normwise, the rank-32 bar of tests/test_mlp_gpu.py."""
    F, H, nh, B = 4, 8, 1, 3
    m = Q.MLP(F, H, nh, P, r, seed=P)
    p = m.get_params()
    p *= 6.0
    m.set_params(p)
    rng = np.random.default_rng(P)
    X = rng.normal(size=(B, F)).astype(np.float32)
    As = np.stack([spd_unit_diag(P, 50 + s) for s in range(B)]).astype(np.float32)
    m.set_data(X, As)
    idx = np.arange(B, dtype=np.int32)
    loss, g = m.loss_grad(idx)
    lo, go = O.mlp_loss_grad(F, H, nh, P, r, oracle_params(m), bf16(X), As.astype(np.float64))
    gb, gob = g[-m.out_dim:], go[-m.out_dim:]
    err = np.max(np.abs(gb - gob)) / np.max(np.abs(gob))
    print(f"P={P} r={r}: loss {loss:.6f} oracle {lo:.6f} bias gradient err {err:.2e}")
    assert abs(loss - lo) <= 1e-2 * max(1.0, abs(lo))
    assert err <= 3.5e-2
    m.close()
