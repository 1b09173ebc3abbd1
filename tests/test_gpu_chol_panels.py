"""Cholesky factors up to 128 columns at the edges of the 16-column panels and of the
kernel's sizes (16, 32, 48, 64, 128), with dead pivots in every place of a panel.
Against LAPACK; tolerances in units of c u times the condition of the scaled factor."""
import numpy as np
import pytest

from test_gpu_dense import _chol

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("c", [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 81, 95, 97,
                               112, 113, 127, 128])
@pytest.mark.parametrize("rows", [60, 3, 1])
def test_factor_inverse_and_condition(c, rows):
    # 60 c rows: Gershgorin's bound from c = 16 down; 3 c, c + 2: the iterations
    rng = np.random.default_rng(c)
    A = rng.standard_normal((rows * c + 2, c)) * np.logspace(0, 4, c)
    G = A.T @ A
    R, T, info, dinfo = _chol(G)
    d = np.sqrt(np.diag(G))
    S = G / np.outer(d, d)
    kappa = np.sqrt(np.linalg.cond(S))
    assert info == 0 and dinfo[2] == 0 and dinfo[3] == pytest.approx(np.max(np.diag(G)), rel=1e-14)
    assert not np.any(np.tril(R, -1)) and not np.any(np.tril(T, -1))
    assert np.max(np.abs(R.T @ R / np.outer(d, d) - S)) < 32 * c * U
    assert np.max(np.abs((T @ R) * d[:, None] / d[None, :] - np.eye(c))) < 64 * c * U * kappa
    assert 0.5 * kappa < dinfo[1] < 1.8 * kappa
    assert np.linalg.norm(R / d) * np.linalg.norm(T * d[:, None]) == pytest.approx(dinfo[0], rel=1e-8)


@pytest.mark.parametrize("c,dead", [(5, 0), (16, 15), (30, 16), (48, 31), (70, 69), (128, 64)])
def test_dead_pivot_and_shift(c, dead):
    rng = np.random.default_rng(c)
    A = rng.standard_normal((8 * c, c)) * np.logspace(0, 4, c)
    G = A.T @ A
    G[dead, :] = 0.0
    G[:, dead] = 0.0
    keep = np.arange(c) != dead
    d = np.sqrt(np.diag(G))[keep]
    R, T, info, dinfo = _chol(G)
    assert info == 1 and dinfo[2] == 1
    assert not np.any(R[dead]) and not np.any(T[:, dead])
    TR = (T @ R)[np.ix_(keep, keep)]
    assert np.max(np.abs(TR * d[:, None] / d[None, :] - np.eye(c - 1))) < 64 * c * U
    shift = 1e-3
    R, T, info, _ = _chol(G, shift=shift, tiny=0.0)
    assert info == 1
    S = G[np.ix_(keep, keep)] / np.outer(d, d) + shift * np.eye(c - 1)
    Rk = R[np.ix_(keep, keep)]
    assert np.max(np.abs(Rk.T @ Rk / np.outer(d, d) - S)) < 32 * c * U


def test_dependent_column_is_dead():
    # the last column lies in the span of two others: its pivot is rounding
    rng = np.random.default_rng(3)
    A = rng.standard_normal((300, 40))
    A[:, 39] = A[:, 0] + 3e-7 * A[:, 1]
    R, T, info, dinfo = _chol(A.T @ A)
    assert info == 1 and dinfo[2] == 1
    assert not np.any(R[39]) and not np.any(T[:, 39])
