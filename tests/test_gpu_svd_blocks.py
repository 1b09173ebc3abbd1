"""The Jacobi SVD over many workgroups at the edges of its block and row
layouts (57 columns is the first count that takes it): one block short or
full, a last block that is empty, rows beside every padding step, and columns
too long for the padded layouts.  Against LAPACK: singular values within
64 sqrt(k) u s0, V orthogonal and A = U S V^T within 64 k u s0."""
import numpy as np
import pytest

from test_gpu_dense import _svd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(57, 57), (64, 64), (65, 65), (80, 80), (81, 81), (128, 97),
                                 (129, 129), (192, 96), (193, 60), (256, 161), (257, 70),
                                 (1300, 58), (5000, 57), (3000, 6)])
@pytest.mark.parametrize("wantV", [True, False])
def test_svd_many_workgroups(m, k, wantV):
    rng = np.random.default_rng(m * 1000 + k)
    A = rng.standard_normal((m, k)) * np.logspace(0, -3, k)
    A[:, k // 3] = 0.0
    s, U, V, iv, Aafter = _svd(A, wantV)
    assert np.array_equal(Aafter, A)
    u = 2.0 ** -53
    sref = np.linalg.svd(A, compute_uv=False)
    assert np.all(np.diff(s) <= 0) and s[-1] == 0.0
    assert np.max(np.abs(s - sref)) < 64 * np.sqrt(k) * u * sref[0]
    assert iv[0] == k - 1 and 1 <= iv[2] < 40
    if wantV:
        assert np.max(np.abs(V.T @ V - np.eye(k))) < 64 * k * u
        assert np.max(np.abs((U * s) @ V.T - A)) < 64 * k * u * sref[0]
