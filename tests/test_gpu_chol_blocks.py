"""Cholesky factors beyond 128 columns (block rows of 128) at the edges of
the blocks: one column over, a full last block, three and four blocks.
Against LAPACK; tolerances in units of c u for well-conditioned scaled Grams
(kappa of the scaled Gram below 10)."""
import numpy as np
import pytest

from test_gpu_dense import _chol

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _gram(c, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((8 * c, c)) * np.logspace(0, 4, c)
    return A.T @ A


@pytest.mark.parametrize("c", [129, 255, 256, 257, 385, 513])
def test_factor_inverse_and_condition(c):
    G = _gram(c, c)
    R, T, info, dinfo = _chol(G)
    d = np.sqrt(np.diag(G))
    assert info == 0 and dinfo[2] == 0 and dinfo[3] == pytest.approx(np.max(np.diag(G)), rel=1e-14)
    assert not np.any(np.tril(R, -1)) and not np.any(np.tril(T, -1))
    S = G / np.outer(d, d)
    assert np.max(np.abs(R.T @ R / np.outer(d, d) - S)) < 32 * c * U
    assert np.max(np.abs((T @ R) * d[:, None] / d[None, :] - np.eye(c))) < 64 * c * U
    kappa = np.sqrt(np.linalg.cond(S))
    assert 0.5 * kappa < dinfo[1] < 1.1 * kappa
    assert np.linalg.norm(R / d) * np.linalg.norm(T * d[:, None]) == pytest.approx(dinfo[0], rel=1e-10)


@pytest.mark.parametrize("c,dead", [(129, 128), (200, 0), (300, 130)])
def test_dead_pivot_and_shift(c, dead):
    G = _gram(c, c)
    G[dead, :] = 0.0
    G[:, dead] = 0.0
    R, T, info, dinfo = _chol(G)
    assert info == 1 and dinfo[2] == 1
    assert not np.any(R[dead]) and not np.any(T[:, dead])
    keep = np.arange(c) != dead
    TR = (T @ R)[np.ix_(keep, keep)]
    d = np.sqrt(np.diag(G))[keep]
    assert np.max(np.abs(TR * d[:, None] / d[None, :] - np.eye(c - 1))) < 64 * c * U
    shift = 1e-3
    R, T, info, _ = _chol(G, shift=shift, tiny=0.0)
    assert info == 1
    S = G[np.ix_(keep, keep)] / np.outer(d, d) + shift * np.eye(c - 1)
    Rk = R[np.ix_(keep, keep)]
    assert np.max(np.abs(Rk.T @ Rk / np.outer(d, d) - S)) < 32 * c * U
