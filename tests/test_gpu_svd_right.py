"""Right singular vectors of a triangular factor (ptt_hip_svd_right) at the
edges of its layouts (32, 48, 64, 96, 128 columns and one more; rank beyond 64
columns goes over many workgroups), for flat, graded, rank-deficient and zero
factors and far magnitudes.  Against LAPACK, in units of k u s0."""
import ctypes as C

import numpy as np
import pytest

import paratt_amd as P
from gpu_util import DevBuf
from test_gpu_dense import _tail_rank

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _right(R, delta=0.0, cap=1000):
    L = P.lib()
    L.ptt_hip_svd_right.argtypes = [C.c_int, C.c_void_p, C.c_long, C.c_void_p, C.c_void_p,
                                    C.c_void_p, C.c_long, C.c_double, C.c_int, C.c_void_p]
    k = R.shape[0]
    r, x = DevBuf(np.asfortranarray(R).ravel(order="F")), DevBuf(np.zeros(k * k))
    s, v = DevBuf(np.full(k, np.nan)), DevBuf(np.full(k * k, np.nan))
    io = DevBuf(np.zeros(8, np.int32), np.int32)
    L.ptt_hip_svd_right(k, r.ptr, k, x.ptr, s.ptr, v.ptr, k, delta, cap, io.ptr)
    L.ptt_hip_sync()
    out = s.get(), v.get().reshape(k, k, order="F"), io.get()
    for b in (r, x, s, v, io):
        b.free()
    return out


def _factor(k, kind):
    rng = np.random.default_rng(k)
    M = rng.standard_normal((k, 4 * k))
    if kind == "graded":
        M = M * np.logspace(0, -12, k)[:, None]
    if kind == "deficient":
        q = max(1, k // 3)
        M = M[:, :q] @ (np.logspace(0, -8, q)[:, None] * rng.standard_normal((q, 4 * k)))
    if kind == "tiny":
        M = M * 1e-200
    return np.linalg.qr(M.T, mode="r")


@pytest.mark.parametrize("kind", ["flat", "graded", "deficient", "tiny"])
@pytest.mark.parametrize("k", [1, 2, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128])
def test_right_vectors(k, kind):
    R = _factor(k, kind)
    s, V, io = _right(R)
    sref = np.linalg.svd(R, compute_uv=False)
    s0 = sref[0]
    assert np.max(np.abs(s - sref)) < 16 * k * U * s0 and np.all(np.diff(s) <= 0)
    nk = int(io[0])
    assert nk == (max(1, k // 3) if kind == "deficient" else k)
    V = V[:, :nk]
    assert np.max(np.abs(V.T @ V - np.eye(nk))) < 16 * k * U
    # L V V^T = L up to the content below the numerical rank
    assert np.max(np.abs(R.T @ V @ V.T - R.T)) < 16 * k * U * s0


@pytest.mark.parametrize("k", [30, 100])
def test_rank_rule(k):
    R = _factor(k, "graded")
    for delta in (1e-3, 1e-7):
        for cap in (k, k // 4):
            s, _, io = _right(R, delta, cap)
            assert io[1] == _tail_rank(s, delta, int(io[0]), cap)


@pytest.mark.parametrize("k", [5, 70])
def test_zero_factor(k):
    s, V, io = _right(np.zeros((k, k)))
    assert not np.any(s) and io[0] == 0 and io[1] == 1
    assert np.linalg.norm(V[:, 0]) == 1.0
