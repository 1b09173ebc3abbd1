"""Eigen-decomposition of Grams whose leading rows are zero or diagonal: no
reflector touches them, so row waves of the tridiagonalisation go idle before the
first one.  Each case runs after a kernel that leaves NaN in the LDS of every CU.
Bars as of the solver's other tests (64 c u of ||G||)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from gpu_util import DevBuf
from test_gpu_syev_merge import _check

pytestmark = pytest.mark.gpu


def _nan_in_lds():
    """The Gram of a 131072 x 128 matrix of NaN: 66 KB of LDS on 256 workgroups."""
    L = P.lib()
    L.ptt_hip_gram.argtypes = [C.c_char, C.c_int, C.c_long, C.c_void_p, C.c_long, C.c_void_p]
    A = DevBuf(np.full(131072 * 128, np.nan))
    G = DevBuf(np.zeros(128 * 128))
    L.ptt_hip_gram(b"T", 128, 131072, A.ptr, 131072, G.ptr)
    L.ptt_hip_sync()
    A.free()
    G.free()


@pytest.mark.parametrize("lead", ["zero", "diagonal"])
@pytest.mark.parametrize("c,k", [(48, 16), (48, 17), (48, 40), (100, 16), (100, 17), (100, 40),
                                 (100, 97), (192, 16), (192, 112), (192, 113), (192, 130)])
def test_leading_rows(c, k, lead):
    rng = np.random.default_rng(1000 * c + k)
    G = np.zeros((c, c))
    M = rng.standard_normal((c - k, 3 * (c - k) + 2))
    G[k:, k:] = M @ M.T
    if lead == "diagonal":
        G[np.arange(k), np.arange(k)] = 1.0 + rng.random(k)
    _nan_in_lds()
    _check(G)


@pytest.mark.parametrize("rx,ry", [(16, 24), (20, 60), (100, 60)])
def test_rounding_of_a_sum_with_weight_zero(rx, ry):
    n = [60] * 4
    x = O.gauss_tt(n, [1] + [rx] * 3 + [1], 1, 0.1)
    y = O.gauss_tt(n, [1] + [ry] * 3 + [1], 2, 0.1)
    z = O.axpby(0.0, x, 1.0, y)
    tol = 1e-9 * O.norm(z)
    ref = O.truncate(z, tol, z.r)
    dz = P.DevTT.from_host(z)
    _nan_in_lds()
    P.truncate(dz, tol, z.r)
    out = O.HostTT(dz.n, dz.r, dz.download_cores())
    assert out.r == ref.r
    assert O.rel_diff(out, ref) < 1e-11
