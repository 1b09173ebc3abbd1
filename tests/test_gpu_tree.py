"""Rounding of low-rank trains by Householder trees (tsqr.hip) where its
layouts change: 1, 15, 16 (one column a lane), 17, 31, 32 columns (two; changed
over to from the Cholesky-QR sweep on an ill-conditioned core), blocks of 128,
256 and 512 rows and one row more, two and three levels, a capped and an
eps-bound cut, numerically rank-deficient sums, wide first cores.  Against the
CPU oracle: identical ranks; trains within 64 d u of each other relative to the
norm where the cut is clean (the oracle's own backward error), plus what the
cut's gap turns (eps * 1e-3)."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from gpu_util import to_host

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _round(z, eps, mr):
    t = P.DevTT.from_host(z)
    P.truncate_rel(t, eps, mr)
    out, stats = to_host(t), P.last_round_stats()
    return out, stats


def _check(z, eps, mr):
    ref = O.truncate(z, eps * O.norm(z), mr)
    out, stats = _round(z, eps, mr)
    assert out.r == ref.r
    assert O.rel_diff(out, ref) < 64 * z.d * U + 1e-3 * eps
    assert stats.norm == pytest.approx(O.norm(z), rel=64 * z.d * U)
    return out, stats


@pytest.mark.parametrize("r", [1, 2, 15, 16])
@pytest.mark.parametrize("n", [8, 9, 16, 17, 32, 33])
def test_rank_deficient_sum_keeps_half(r, n):
    # x + 1e-3 x' with x' = x: formal rank 2 r, numerical rank r (ranks of 1 to
    # 32 columns; rows r n from one block to three levels)
    x = O.gauss_tt([n] * 5, [1, r, r, r, r, 1], 7 * r + n)
    z = O.axpby(1.0, x, 1e-3, x)
    out, _ = _check(z, 1e-10, [1, 64, 64, 64, 64, 1])
    assert out.r == [1] + [min(r, n ** min(k, 5 - k)) for k in range(1, 5)] + [1]


@pytest.mark.parametrize("r,n", [(8, 16), (16, 8), (16, 32), (15, 35), (16, 300), (5, 1700)])
@pytest.mark.parametrize("cap", [0, 3])
def test_small_update_and_cap(r, n, cap):
    d = 4
    x = O.gauss_tt([n] * d, [1] + [r - r // 3] * (d - 1) + [1], 3)
    y = O.gauss_tt([n] * d, [1] + [r // 3] * (d - 1) + [1], 4)
    z = O.axpby(1.0, x, 1e-12, y)
    mr = [1] + [cap or 64] * (d - 1) + [1]
    out, stats = _round(z, 1e-8, mr)
    ref = O.truncate(z, 1e-8 * O.norm(z), mr)
    assert out.r == ref.r
    # a cap among a random train's singular values turns the subspace by
    # u s0 / gap; gaps of its few hundred values stay above 1e-5 s0
    assert O.rel_diff(out, ref) < 64 * d * U * (1e5 if cap else 1.0) + 1e-11
    assert max(stats.ltr_cholqr_passes[:d - 1]) == 0  # no Cholesky-QR pass was taken


@pytest.mark.parametrize("r", [9, 16])
def test_changes_over_at_the_first_ill_conditioned_core(r):
    # ranks 2 r = 18, 32: Cholesky-QR starts the sweep, the copies' cores are
    # rank-deficient
    x = O.gauss_tt([40, 64, 64, 50, 40], [1, r, r, r, r, 1], 5)
    z = O.axpby(1.0, x, 1e-3, x)
    out, stats = _check(z, 1e-9, [1, 64, 64, 64, 64, 1])
    assert list(stats.ltr_cholqr_passes[1:4]) == [0, 0, 0]


def test_views_and_many_modes():
    import ctypes as C
    # the raw-array entry point (borrowed cores) and more modes than the
    # statistics hold
    d = 70
    x = O.gauss_tt([3] * d, [1] + [4] * (d - 1) + [1], 6)
    z = O.axpby(1.0, x, 1e-3, x)
    ref = O.truncate(z, 1e-9 * O.norm(z), z.r)
    t = P.DevTT.from_host(z)
    tt = t.tt.contents
    mr = (C.c_int * (d + 1))(*([1] + [8] * (d - 1) + [1]))
    L = P.lib()
    L.pattacTruncate.argtypes = [C.c_int, C.c_int, C.POINTER(C.c_int), C.POINTER(C.c_int),
                                 C.POINTER(C.c_void_p), C.POINTER(C.c_int), C.c_double, C.c_double,
                                 C.c_char, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    before = [tt.coreList[k] for k in range(d)]
    L.pattacTruncate(0, d, tt.dim, tt.ttRank, tt.coreList, mr, 1e-9 * O.norm(z), 0.0, b"R", None,
                     None, None, None)
    assert [tt.coreList[k] for k in range(d)] == before
    out = to_host(t)
    assert out.r == ref.r and O.rel_diff(out, ref) < 64 * d * U + 1e-12
