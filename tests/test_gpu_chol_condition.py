"""The condition estimate of Cholesky factors beyond 128 columns is that of ten power
iterations a side, on either side of the size up to which the matrix is held in
registers.  Against the same iterations in numpy; both round to some hundred u, the
difference between six iterations and ten is 0.3% to 7% on these matrices."""
import numpy as np
import pytest

from test_gpu_dense import _chol

pytestmark = pytest.mark.gpu


def _power(apply, c, period, its=10):
    x = 1.0 + 0.01 * (np.arange(c) % period)
    for _ in range(its):
        y = apply(x)
        ratio = np.linalg.norm(y) / np.linalg.norm(x)
        x = y / np.linalg.norm(y)
    return ratio


@pytest.mark.parametrize("kind", ["paired", "nearly_square"])
@pytest.mark.parametrize("c", [130, 192, 193, 256])
def test_ten_iterations_a_side(c, kind):
    rng = np.random.default_rng(c)
    A = rng.standard_normal((8 * c if kind == "paired" else c + 40, c))
    if kind == "paired":
        A[:, 1::2] = A[:, ::2][:, : c // 2] + 0.1 * A[:, 1::2]
    G = A.T @ A
    d = np.sqrt(np.diag(G))
    S = G / np.outer(d, d)
    T = np.linalg.inv(np.linalg.cholesky(S)).T
    ref = np.sqrt(_power(lambda x: S @ x, c, 7) * _power(lambda x: T @ (T.T @ x), c, 5))
    six = np.sqrt(_power(lambda x: S @ x, c, 7, 6) * _power(lambda x: T @ (T.T @ x), c, 5, 6))
    assert abs(six - ref) > 1e-3 * ref
    info = _chol(G)
    assert info[2] == 0
    assert abs(info[3][1] - ref) <= 1e-9 * ref
