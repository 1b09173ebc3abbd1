"""ptt_hip_syev_gram from 129 to 192 rows: two tile rows a wave in the
tridiagonalisation, merges of 128 rows below the top one, reflectors staged in
parts.  The edges of its blocks, deflating and graded spectra, and the rank rule;
bars as of the solver's other tests (64 c u of ||G||)."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from test_gpu_syev import syev
from test_gpu_syev_merge import _check, _spectrum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["gauss", "clusters", "flat", "far"])
@pytest.mark.parametrize("c", [129, 130, 144, 145, 160, 161, 190, 191, 192])
def test_edges(c, kind):
    rng = np.random.default_rng(100 * c + len(kind))
    Q, _ = np.linalg.qr(rng.standard_normal((c, c)))
    G = (Q * _spectrum(kind, c, rng)) @ Q.T
    _check((G + G.T) / 2)


@pytest.mark.parametrize("c,cut", [(192, 64), (192, 128), (160, 96), (150, 33), (192, 191)])
def test_zero_couplings(c, cut):
    rng = np.random.default_rng(c + cut)
    G = np.zeros((c, c))
    for a, b in ((0, cut), (cut, c)):
        M = rng.standard_normal((b - a, 3 * (b - a) + 2))
        G[a:b, a:b] = M @ M.T
    _check(G)


@pytest.mark.parametrize("c", [129, 180, 192])
def test_diagonal_and_rank_rule(c):
    d = np.logspace(0, -8, c)[::-1]
    sig, U, iout, dinfo = syev(np.diag(d), delta=1e-3, cap=c)
    ref = np.sqrt(np.sort(d)[::-1])
    assert np.max(np.abs(sig - ref)) <= 1e-15
    tail = np.sqrt(np.cumsum(ref[::-1] ** 2))[::-1]
    assert iout[0] == c and iout[1] == max(1, int(np.sum(tail >= 1e-3)))
    assert dinfo[6] == 1.0 and dinfo[7] == pytest.approx(d.sum(), rel=1e-14)
    assert syev(np.diag(d), delta=1e-3, cap=70)[2][1] == 70


@pytest.mark.parametrize("rx,ry,cap", [(80, 60, 90), (100, 92, 100), (66, 63, 0)])
def test_rounding_matches_oracle(rx, ry, cap):
    n = [40] * 4
    x = O.gauss_tt(n, [1] + [rx] * 3 + [1], 1, 1.0 / np.sqrt(40 * rx))
    y = O.gauss_tt(n, [1] + [ry] * 3 + [1], 2, 1.0 / np.sqrt(40 * ry))
    z = O.axpby(1.0, x, 1.0, y)
    caps = [1] + [cap or rx + ry] * 3 + [1]
    tol = 1e-8 * O.norm(z)
    ref = O.truncate(z, tol, caps)
    dz = P.DevTT.from_host(z)
    P.truncate(dz, tol, caps)
    out = O.HostTT(dz.n, dz.r, dz.download_cores())
    assert out.r == ref.r
    # 1e-12 of the norm beside a cut between nearly tied singular values
    assert O.rel_diff(out, ref) < 1e-11
