"""Divide and conquer of ptt_hip_syev_gram at the edges of its blocks (leaves of
two rows, workgroups of 32, merges of 64 and 128) and on spectra that deflate:
clusters (rotations at many neighbouring poles), zero couplings (blocks that are
not merged) and one far eigenvalue.  Same bars as the solver's other tests, which
are the Gram's own rounding: 64 c u of ||G|| for eigenvalues and residual, 64 c u
for orthogonality."""
import numpy as np
import pytest

from test_gpu_syev import U64, syev

pytestmark = pytest.mark.gpu


def _spectrum(kind, c, rng):
    if kind == "gauss":
        return np.sort(rng.random(c) + 0.1)
    if kind == "clusters":  # groups of nearly equal values, some exactly equal
        v = np.repeat(np.linspace(1.0, 0.2, (c + 6) // 7), 7)[:c]
        return v * (1.0 + 1e-15 * rng.integers(0, 3, c))
    if kind == "flat":
        return 1.0 + 1e-3 * rng.random(c)
    return np.r_[1e6, rng.random(c - 1)]  # far


@pytest.mark.parametrize("kind", ["gauss", "clusters", "flat", "far"])
@pytest.mark.parametrize("c", [2, 4, 6, 17, 31, 32, 34, 63, 66, 96, 97, 126])
def test_merge_edges(c, kind):
    rng = np.random.default_rng(100 * c + len(kind))
    Q, _ = np.linalg.qr(rng.standard_normal((c, c)))
    G = (Q * _spectrum(kind, c, rng)) @ Q.T
    _check((G + G.T) / 2)


@pytest.mark.parametrize("c,cut", [(64, 32), (64, 33), (128, 64), (128, 31), (100, 96), (33, 32)])
def test_zero_couplings(c, cut):
    """Two blocks that do not touch: the couplings that part them are zero."""
    rng = np.random.default_rng(c + cut)
    G = np.zeros((c, c))
    for a, b in ((0, cut), (cut, c)):
        M = rng.standard_normal((b - a, 3 * (b - a) + 2))
        G[a:b, a:b] = M @ M.T
    _check(G)


def _check(G):
    c = G.shape[0]
    sig, U, iout, _ = syev(G)
    ref = np.maximum(np.sort(np.linalg.eigvalsh(G))[::-1], 0.0)
    bar = 64 * c * U64
    lam = sig ** 2
    assert np.all(np.diff(sig) <= 0)
    assert np.max(np.abs(lam - ref)) <= bar * ref[0]
    assert np.linalg.norm(G @ U - U * lam) <= bar * ref[0]
    assert np.linalg.norm(U.T @ U - np.eye(c)) <= bar
