"""Singular values and right vectors of L = R^T from approximate left ones
(ptt_hip_svd_right_from), the eigenvectors of the Gram R^T R as the Gram route leaves
them: at the edges of its paths (64 columns on one workgroup, 128, 192), V in
place of U, flat and graded factors and far magnitudes.  Against LAPACK, in units
of k u s0 as the other starts."""
import ctypes as C

import numpy as np
import pytest

import paratt_amd as P
from gpu_util import DevBuf
from test_gpu_dense import _tail_rank

pytestmark = pytest.mark.gpu
U64 = 2.0 ** -53


def _right_from(R, U, delta=0.0, cap=1000):
    L = P.lib()
    L.ptt_hip_svd_right_from.argtypes = [C.c_int, C.c_void_p, C.c_long, C.c_void_p, C.c_long,
                                         C.c_void_p, C.c_void_p, C.c_void_p, C.c_long, C.c_double,
                                         C.c_int, C.c_void_p]
    k = R.shape[0]
    r, x = DevBuf(np.asfortranarray(R).ravel(order="F")), DevBuf(np.zeros(k * k))
    s, v = DevBuf(np.full(k, np.nan)), DevBuf(np.asfortranarray(U).ravel(order="F"))
    io = DevBuf(np.zeros(8, np.int32), np.int32)
    L.ptt_hip_svd_right_from(k, r.ptr, k, v.ptr, k, x.ptr, s.ptr, v.ptr, k, delta, cap, io.ptr)
    L.ptt_hip_sync()
    out = s.get(), v.get().reshape(k, k, order="F"), io.get()
    for b in (r, x, s, v, io):
        b.free()
    return out


def _factor(k, kind):
    rng = np.random.default_rng(k)
    M = rng.standard_normal((k, 4 * k))
    if kind == "graded":
        M = M * np.logspace(0, -6, k)[:, None]
    if kind == "tiny":
        M = M * 1e-120
    return np.linalg.qr(M.T, mode="r")


@pytest.mark.parametrize("kind", ["flat", "graded", "tiny"])
@pytest.mark.parametrize("k", [1, 2, 31, 33, 63, 64, 65, 128, 129, 161, 192])
def test_right_vectors(k, kind):
    R = _factor(k, kind)
    S = R / np.max(np.abs(R))
    _, U = np.linalg.eigh(S.T @ S)
    s, V, io = _right_from(R, U)
    sref = np.linalg.svd(R, compute_uv=False)
    assert np.max(np.abs(s - sref)) < 16 * k * U64 * sref[0] and np.all(np.diff(s) <= 0)
    assert io[0] == k
    assert np.max(np.abs(V.T @ V - np.eye(k))) < 16 * k * U64
    # L V = (left vectors) Sigma: orthogonal columns, up to rounding of s0
    B = R.T @ V
    D = B.T @ B
    assert np.max(np.abs(D - np.diag(np.diag(D)))) < 16 * k * U64 * sref[0] ** 2
    for delta, cap in ((1e-3 * sref[0], k), (1e-3 * sref[0], max(1, k // 4))):
        s, _, io = _right_from(R, U, delta, cap)
        assert io[1] == _tail_rank(s, delta, int(io[0]), cap)


def test_any_orthogonal_start():
    """A start that approximates nothing only costs sweeps."""
    for k in (40, 90, 150):
        R = _factor(k, "flat")
        Q, _ = np.linalg.qr(np.random.default_rng(1).standard_normal((k, k)))
        s, V, io = _right_from(R, Q)
        sref = np.linalg.svd(R, compute_uv=False)
        assert np.max(np.abs(s - sref)) < 16 * k * U64 * sref[0]
        assert np.max(np.abs(V.T @ V - np.eye(k))) < 16 * k * U64
