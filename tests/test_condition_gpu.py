"""Condition numbers of the drop-in API (Householder tridiagonalisation and multisection on the
GPU) against numpy's singular values, at the sizes where the kernel's row split changes.  Bar:
a backward-stable eigenvalue is off by at most P eps ||A||, i.e. kappa by P eps kappa relative
(kappa^2 for a general matrix, whose singular values come from M^H M), plus float rounding."""
import ctypes

import numpy as np
import pytest

import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu


def _kappa(M):
    L = Q.lib()
    f = L.compute_complex_matrix_condition_number
    f.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.POINTER(ctypes.c_float)]
    f.restype = ctypes.c_bool
    M = np.ascontiguousarray(M, np.complex64)
    k = ctypes.c_float()
    assert f(M.ctypes.data, len(M), ctypes.byref(k))
    return k.value


def _hermitian(P, ev, seed):
    rng = np.random.default_rng(seed)
    V, _ = np.linalg.qr(rng.normal(size=(P, P)) + 1j * rng.normal(size=(P, P)))
    M = ((V * ev) @ V.conj().T).astype(np.complex64)
    return np.tril(M, -1) + np.tril(M, -1).conj().T + np.diag(M.diagonal().real)


def _check(M, general=False):
    sv = np.linalg.svd(M.astype(np.complex128), compute_uv=False)
    ref = sv.max() / sv.min()
    eps = np.finfo(np.float64).eps
    assert abs(_kappa(M) - ref) <= ref * (1e-6 + len(M) * eps * ref ** (2 if general else 1))


@pytest.mark.parametrize("P", [2, 3, 31, 64, 65, 96, 128, 129, 171, 342, 513])
def test_condition_number_hermitian(P):
    _check(_hermitian(P, 0.25 * np.logspace(-4, 0, P), P))
    ev = np.linspace(-1.0, 1.0, P) + 0.3 / P               # both signs, the smallest either side of zero
    _check(_hermitian(P, ev, P + 1))
    _check(_hermitian(P, -ev, P + 2))


@pytest.mark.parametrize("P", [2, 5, 66, 130])
def test_condition_number_general(P):
    rng = np.random.default_rng(P)
    U, _ = np.linalg.qr(rng.normal(size=(P, P)) + 1j * rng.normal(size=(P, P)))
    V, _ = np.linalg.qr(rng.normal(size=(P, P)) + 1j * rng.normal(size=(P, P)))
    _check(((U * np.logspace(-2, 0, P)) @ V).astype(np.complex64), general=True)


def test_condition_number_zero_rows_and_diagonals():
    assert _kappa(np.eye(1)) == 1.0
    assert _kappa(np.diag([4.0, 0.0, -2.0, 0.5])) == 8.0    # exact zeros are not counted
    assert _kappa(np.zeros((3, 3))) == 0.0                  # no nonzero value at all: 0 / inf
    M = np.zeros((70, 70), np.complex64)                     # a parameter without effect: an exact zero row
    keep = [i for i in range(70) if i not in (0, 13, 64)]
    B = _hermitian(67, 0.25 * np.logspace(-3, 0, 67), 5)
    M[np.ix_(keep, keep)] = B
    sv = np.abs(np.linalg.eigvalsh(B.astype(np.complex128)))
    assert abs(_kappa(M) - sv.max() / sv.min()) <= 1e-6 * sv.max() / sv.min()
    assert np.isinf(_kappa(np.ones((40, 40)))) or _kappa(np.ones((40, 40))) > 1e13   # rank one


def _extremes(A):
    """qgtl_hip_herm_extremes_c128 itself, A one component: smallest, largest, smallest positive, largest
    negative; smallest size, bound."""
    L, vp, ip = Q.lib(), ctypes.c_void_p, ctypes.c_int
    A = np.ascontiguousarray(A, np.complex128)
    out = np.full(6, 7.0)
    L.qgtl_hip_herm_extremes_c128.argtypes = [vp, vp, ip, vp, ip, ip, vp]
    for f in ("h2d", "d2h"):
        getattr(L, "qgtl_hip_" + f).argtypes = [vp, vp, ctypes.c_size_t]
    L.qgtl_hip_malloc.argtypes = [ctypes.POINTER(vp), ctypes.c_size_t]
    L.qgtl_hip_free.argtypes = [vp]
    Q.init()
    d = [vp() for _ in range(3)]
    for p, n in zip(d, (A.nbytes, A.nbytes, out.nbytes)):
        assert L.qgtl_hip_malloc(ctypes.byref(p), n) == 0
    assert L.qgtl_hip_h2d(d[0], A.ctypes.data, A.nbytes) == 0
    assert L.qgtl_hip_herm_extremes_c128(d[0], d[1], len(A), None, 1, len(A), d[2]) == 0
    assert L.qgtl_hip_d2h(out.ctypes.data, d[2], out.nbytes) == 0 and L.qgtl_hip_sync() == 0
    for p in d:
        L.qgtl_hip_free(p)
    return out


@pytest.mark.parametrize("P", [6, 64, 100, 140])
@pytest.mark.parametrize("scale", [1.0, 1e-62])
def test_extremes_of_a_tiny_rank_deficient_matrix(P, scale):
    """M^H M of entries near 1e-31, of rank 2: the columns left after two steps are rounding, 1e-78, whose
    reflector's tau is near 1e156.  The bar is backward stability, P eps ||A|| (times 4)."""
    rng = np.random.default_rng(P)
    V = rng.normal(size=(P, 2)) + 1j * rng.normal(size=(P, 2))
    A = V @ V.conj().T
    ev = np.linalg.eigvalsh(A)
    lo, hi = _extremes(A * scale)[:2] / scale
    assert abs(hi - ev[-1]) <= 4 * P * np.finfo(float).eps * ev[-1]
    assert abs(lo - ev[0]) <= 4 * P * np.finfo(float).eps * ev[-1]


def _coupled(P, rng, general):
    """A P x P block all of whose indices are coupled, condition number about 100."""
    U, _ = np.linalg.qr(rng.normal(size=(P, P)) + 1j * rng.normal(size=(P, P)))
    V = U
    if general:
        V, _ = np.linalg.qr(rng.normal(size=(P, P)) + 1j * rng.normal(size=(P, P)))
    B = (U * np.logspace(-2, 0, P)) @ V.conj().T
    return B if general else 0.5 * (B + B.conj().T)


# sizes of the blocks: all within one kernel form, and across its limits of 64 and 128
@pytest.mark.parametrize("sizes", [(2, 2), (5, 3, 4), (50, 40), (90, 33, 20), (140, 20)])
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("scales", [(1e5, 1e-11), (1.0, 1e-31), (1.0, 1e-7), (1e5, 1e-6)])
@pytest.mark.parametrize("mixed", [False, True])
def test_condition_number_of_decoupled_blocks(sizes, general, scales, mixed):
    """Blocks that no entry couples keep their own accuracy however small they are beside the others
    (and wherever their indices stand): the extremes are those of each block by itself."""
    rng = np.random.default_rng(sum(sizes))
    blocks = [_coupled(n, rng, general) * scales[i % 2] for i, n in enumerate(sizes)]
    blocks = [b.astype(np.complex64) for b in blocks]
    if not general:
        blocks = [np.tril(b, -1) + np.tril(b, -1).conj().T + np.diag(b.diagonal().real) for b in blocks]
    P = sum(sizes) + 1                                          # and a row and column of zeros
    M = np.zeros((P, P), np.complex64)
    at = np.arange(P)
    if mixed:
        at = rng.permutation(P)
    o = 0
    for b in blocks:
        i = at[o:o + len(b)]
        M[np.ix_(i, i)] = b
        o += len(b)
    sv = np.concatenate([np.linalg.svd(b.astype(np.complex128), compute_uv=False) for b in blocks])
    ref = sv.max() / sv.min() if sv.min() > 1e-15 else np.inf   # QGTL's rule: 1e-15 is zero
    k = _kappa(M)
    assert k == ref if np.isinf(ref) else abs(k - ref) <= 2e-6 * ref


@pytest.mark.parametrize("P,rank", [(2, 1), (3, 2), (40, 1), (64, 40), (70, 69), (131, 100)])
@pytest.mark.parametrize("scale", [1.0, 1e5])
def test_condition_number_of_coupled_singular_matrices(P, rank, scale):
    """Singular matrices: the smallest nonzero value is rounding, or an exact zero is left out, as the
    eigenvalues of the full decomposition have it."""
    rng = np.random.default_rng(P)
    V = rng.integers(-3, 4, size=(P, rank)) * (1.0 + 0j)
    V[0] = 1.0
    if rank == 1:
        V[:] = 1.0                                              # all entries equal
    M = ((V @ V.conj().T) * scale).astype(np.complex64)
    sv = np.abs(Q.hermitian_eig(M.astype(np.complex128))[0])
    smin = sv[sv > 0].min()
    assert _kappa(M) == (np.float32(sv.max() / smin) if smin > 1e-15 else np.inf)


@pytest.mark.parametrize("P", [2, 40, 64, 100, 140])
def test_condition_number_of_a_nearly_hermitian_matrix(P):
    """Triangles that differ by rounding (here 5e-7 of the largest entry; up to 1e-6 counts as Hermitian):
    the singular values are those of the Hermitian part up to squares, not those of one triangle."""
    rng = np.random.default_rng(P)
    M = _hermitian(P, 0.25 * np.logspace(-3, 0, P), P)
    E = 5e-7 * np.abs(M).max() * rng.choice([-1.0, 1.0], size=(P, P))
    M = (M + np.tril(E, -1)).astype(np.complex64).astype(np.complex128)
    ev = np.linalg.eigvalsh(0.5 * (M + M.conj().T))
    ref = np.abs(ev).max() / np.abs(ev).min()
    assert abs(_kappa(M) - ref) <= ref * (1e-6 + P * np.finfo(np.float64).eps * ref)
