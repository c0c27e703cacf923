"""The complex LU solve (pivoted, batched) on both sides of the sizes where its kernel changes, against
its own residual: partial pivoting keeps ||A x - b|| within about P eps ||A|| ||x|| for matrices
without exceptional growth, here with a factor of 4."""
import ctypes

import numpy as np
import pytest

import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


def _solve(A, b):
    L = Q.lib()
    batch, P = b.shape
    A, b = np.ascontiguousarray(A, np.complex128), np.ascontiguousarray(b, np.complex128)
    x, st = np.zeros_like(b), np.full(batch, 7, np.int32)
    vp = ctypes.c_void_p
    L.qgtl_hip_lu_solve_c128.argtypes = [vp, vp, vp, vp, ctypes.c_int, ctypes.c_int, vp]
    for f in ("h2d", "d2h"):
        getattr(L, "qgtl_hip_" + f).argtypes = [vp, vp, ctypes.c_size_t]
    L.qgtl_hip_malloc.argtypes = [ctypes.POINTER(vp), ctypes.c_size_t]
    L.qgtl_hip_free.argtypes = [vp]
    Q.init()
    d = [vp() for _ in range(5)]
    for p, n in zip(d, (A.nbytes, b.nbytes, b.nbytes, 4 * b.size, st.nbytes)):
        assert L.qgtl_hip_malloc(ctypes.byref(p), n) == 0
    assert L.qgtl_hip_h2d(d[0], A.ctypes.data, A.nbytes) == 0 and L.qgtl_hip_h2d(d[1], b.ctypes.data, b.nbytes) == 0
    assert L.qgtl_hip_lu_solve_c128(d[0], d[1], d[2], d[3], P, batch, d[4]) == 0
    assert L.qgtl_hip_d2h(x.ctypes.data, d[2], x.nbytes) == 0 and L.qgtl_hip_d2h(st.ctypes.data, d[4], st.nbytes) == 0
    assert L.qgtl_hip_sync() == 0
    for p in d:
        L.qgtl_hip_free(p)
    return x, st


SIZES = [1, 2, 3, 15, 16, 17, 63, 64, 65, 96, 127, 128, 129, 150]


@pytest.mark.parametrize("P", SIZES)
def test_random_systems(P):
    rng = np.random.default_rng(P)
    A = rng.normal(size=(3, P, P)) + 1j * rng.normal(size=(3, P, P))
    A[1] *= np.exp(3 * rng.normal(size=(P, 1)))       # rows of very different size: many exchanges
    b = rng.normal(size=(3, P)) + 1j * rng.normal(size=(3, P))
    x, st = _solve(A, b)
    assert (st == 0).all()
    for k in range(3):
        r = np.linalg.norm(A[k] @ x[k] - b[k])
        assert r <= 4 * P * np.finfo(float).eps * (np.linalg.norm(A[k]) * np.linalg.norm(x[k]) + np.linalg.norm(b[k]))


@pytest.mark.parametrize("P", SIZES[1:])
def test_ties_and_exact_permutations(P):
    """Entries of equal size in every column (the first row wins) and a permutation matrix: exact."""
    rng = np.random.default_rng(100 + P)
    perm = rng.permutation(P)
    A = np.zeros((2, P, P), complex)
    A[0, np.arange(P), perm] = 1j
    A[1] = np.tril(np.ones((P, P)))                   # |a| = 1 throughout the columns
    b = (1.0 + np.arange(2 * P)).reshape(2, P) + 0j
    x, st = _solve(A, b)
    assert (st == 0).all()
    want = np.zeros(P, complex)
    want[perm] = b[0] / 1j
    assert np.array_equal(x[0], want)
    assert np.array_equal(x[1], np.concatenate([b[1][:1], np.diff(b[1])]))


@pytest.mark.parametrize("P", [2, 16, 64, 65, 128, 129])
def test_singular_reported(P):
    rng = np.random.default_rng(7)
    A = rng.normal(size=(2, P, P)) + 0j
    A[0, :, P // 2 - 1] = 0.0                         # a zero column before the last
    x, st = _solve(A, np.ones((2, P)))
    assert st[0] == -1 and st[1] == 0 and np.allclose(A[1] @ x[1], 1.0)
