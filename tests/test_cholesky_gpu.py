"""Blocked Cholesky solve at the edges of its column blocks, panel sizes and batches, against
numpy in FP64.  Bar: backward stability, ||(A + lambda I) x - b|| <= 8 P eps ||A + lambda I|| ||x||."""
import numpy as np
import pytest

import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


def _spd(P, seed, lo=1e-6):
    rng = np.random.default_rng(seed)
    V, _ = np.linalg.qr(rng.normal(size=(P, P)))
    A = (V * (0.25 * np.logspace(np.log10(lo), 0, P))) @ V.T
    return 0.5 * (A + A.T), rng.normal(size=P)


def _residual_ok(A, x, b):
    r = np.linalg.norm(A @ x - b)
    assert r <= 8 * len(b) * np.finfo(np.float64).eps * np.linalg.norm(A, 2) * np.linalg.norm(x), r


@pytest.mark.parametrize("P", [1, 2, 4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 192, 255, 256, 257, 511, 512, 513, 1023, 1024])
@pytest.mark.parametrize("noalloc", [False, True])
def test_cholesky_sizes(P, noalloc):
    A, b = _spd(P, P)
    lam = 1e-5
    if noalloc:
        import ctypes
        L = Q.lib()
        L.qgtl_solve_f64_noalloc.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p,
                                             ctypes.c_double, ctypes.c_int, ctypes.c_double, ctypes.c_int,
                                             ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p,
                                             ctypes.c_void_p]
        x = np.zeros(P)
        rc = L.qgtl_solve_f64_noalloc(P, 1, A.ctypes.data, b.ctypes.data, lam, Q.SOLVE_CHOLESKY, 0.0, 1, None, None, 0,
                                      x.ctypes.data, None)
        assert rc == 0
    else:
        x, info = Q.solve(A, b, lam, Q.SOLVE_CHOLESKY)
        assert info["status"] == 0
    _residual_ok(A + lam * np.eye(P), x, b)


@pytest.mark.parametrize("P,batch", [(3, 50), (20, 300), (40, 60), (100, 7), (300, 3)])
def test_cholesky_batch_with_one_indefinite(P, batch):
    """Each system has its own workgroup and status: the one that is not positive definite (a
    negative last pivot, found in the last column block) fails alone."""
    A = np.stack([_spd(P, 10 + i)[0] for i in range(batch)])
    b = np.stack([_spd(P, 10 + i)[1] for i in range(batch)])
    bad = batch // 2
    A[bad, P - 1, P - 1] -= 1.0
    x, info = Q.solve(A, b, 0.0, Q.SOLVE_CHOLESKY, check=False)
    for i in range(batch):
        assert info[i]["status"] == (-1 if i == bad else 0)
        if i != bad:
            _residual_ok(A[i], x[i], b[i])


def test_cholesky_infinite_pivot():
    """An infinite diagonal entry pins its unknown to zero."""
    A, b = _spd(40, 3)
    A[35, 35] = np.inf
    x, info = Q.solve(A, b, 0.0, Q.SOLVE_CHOLESKY)
    keep = np.arange(40) != 35
    assert x[35] == 0.0
    _residual_ok(A[np.ix_(keep, keep)], x[keep], b[keep])
