"""The Kaporin loss kernel itself (qgtl_hip_kaporin, no network around it) against its formulas in
numpy FP64, at the edges of its rank forms, row tiles and vector loads.

Bar: the kernel computes in FP64 throughout, so the loss keeps 16 (r + 1) eps times the size of
its terms, and a gradient entry is one rounding to fp32 (2^-24 of itself) of a value that is off by as
little of the largest entry of its kind (P = 1: of the terms that cancel)."""
import ctypes

import numpy as np
import pytest

import quantum_geometric_tensor_amd as Q

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _kernel(P, r, Y, As, idx, scale):
    L, vp, ip = Q.lib(), ctypes.c_void_p, ctypes.c_int
    B = len(idx)
    loss, dY = np.zeros(B), np.zeros_like(Y)
    L.qgtl_hip_kaporin.argtypes = [ip, ip, ip, vp, vp, vp, vp, vp, ctypes.c_float]
    for f in ("h2d", "d2h"):
        getattr(L, "qgtl_hip_" + f).argtypes = [vp, vp, ctypes.c_size_t]
    L.qgtl_hip_malloc.argtypes = [ctypes.POINTER(vp), ctypes.c_size_t]
    L.qgtl_hip_free.argtypes = [vp]
    Q.init()
    d = [vp() for _ in range(5)]
    for p, a in zip(d, (Y, As, idx, loss, dY)):
        assert L.qgtl_hip_malloc(ctypes.byref(p), a.nbytes) == 0
    for p, a in zip(d[:3], (Y, As, idx)):
        assert L.qgtl_hip_h2d(p, a.ctypes.data, a.nbytes) == 0
    assert L.qgtl_hip_kaporin(P, r, B, d[0], d[1], d[2], d[3], d[4], scale) == 0
    for p, a in ((d[3], loss), (d[4], dY)):
        assert L.qgtl_hip_d2h(a.ctypes.data, p, a.nbytes) == 0
    assert L.qgtl_hip_sync() == 0
    for p in d:
        L.qgtl_hip_free(p)
    return loss, dY


def _reference(P, r, y, A, scale):
    y, A = y.reshape(P, 1 + r).astype(np.float64), A.astype(np.float64)
    s, u = y[:, 0], y[:, 1:] / np.sqrt(P)
    Au = A @ u
    tr = (np.exp(s) * A.diagonal()).sum() + (u * Au).sum()
    W = np.eye(r) + u.T @ (np.exp(-s)[:, None] * u)
    Wi = np.linalg.inv(W)
    loss = P * np.log(tr / P) - s.sum() - np.linalg.slogdet(W)[1]
    size = P * abs(np.log(tr / P)) + np.abs(s).sum() + (r * np.log(np.linalg.norm(W, 2)) if r else 0.0) + P
    g = P / tr
    uW = u @ Wi
    ds = g * np.exp(s) * A.diagonal() - 1.0 + np.exp(-s) * (uW * u).sum(1)
    du = (2 * g * Au - 2 * np.exp(-s)[:, None] * uW) / np.sqrt(P)
    terms = scale * ((g * np.exp(s) * A.diagonal()).max() + 1.0)   # what ds is the difference of
    return loss, size, scale * ds, scale * du, terms


@pytest.mark.parametrize("P,r", [(1, 0), (1, 1), (3, 2), (15, 15), (16, 16), (17, 17), (64, 0), (64, 31), (65, 32),
                                 (127, 16), (128, 16), (129, 16), (191, 8), (192, 8), (256, 32), (300, 27), (481, 17),
                                 (512, 16), (1023, 8), (1024, 8), (1024, 0)])
def test_loss_and_gradient(P, r):
    rng = np.random.default_rng(100 * P + r)
    F = rng.normal(size=(4, P, 2 * P))
    As = (F @ F.transpose(0, 2, 1) / (2 * P)).astype(np.float32)
    As = (As + As.transpose(0, 2, 1)) * np.float32(0.5)
    idx = np.array([3, 0, 1], np.int32)
    Y = rng.normal(size=(3, P * (1 + r))).astype(np.float32)
    Y[1] *= 3.0                                        # W far from the identity
    scale = np.float32(1.0 / 3.0)
    loss, dY = _kernel(P, r, Y, As, idx, scale)
    for b in range(3):
        ref, size, ds, du, terms = _reference(P, r, Y[b], As[idx[b]], float(scale))
        assert abs(loss[b] - ref) <= 16 * (r + 1) * EPS * size
        got = dY[b].reshape(P, 1 + r)
        for mine, want in ((got[:, :1], ds[:, None]), (got[:, 1:], du)):
            if want.size:
                assert np.all(np.abs(mine - want) <= 2.0 ** -24 * (1.001 * np.abs(want) + np.abs(want).max())
                              + 16 * (r + 1) * EPS * terms)
