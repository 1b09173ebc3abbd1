"""NaN and infinities in a Gram given to the eigensolver, and in trains that are
rounded by each of the routes: every call returns with ranks in their range, a value
that is not finite stays visible in the result, and the next rounding is as exact as
ever."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from gpu_util import to_host
from test_gpu_syev import syev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("c", [1, 5, 32, 33, 64, 100, 128, 129, 192])
def test_eigensolver(c, bad):
    rng = np.random.default_rng(c)
    M = rng.standard_normal((c, 3 * c))
    for i, j in {(0, 0), (0, c - 1), (c // 2, c // 2)}:
        G = M @ M.T
        G[i, j] = G[j, i] = bad
        sig, U, iout, _ = syev(G, cap=c)
        assert np.all(np.isnan(sig)) and iout[0] == 0 and iout[1] == 1
        assert np.all(np.isfinite(U))
    G = np.full((c, c), bad)
    sig, _, iout, _ = syev(G, cap=c)
    assert np.all(np.isnan(sig)) and iout[1] == 1


# trees; the two routes of 17 to 32 columns; Gram route to 128 and to 192 rows;
# Jacobi beyond; a last bond with more rows than columns
@pytest.mark.parametrize("n,r", [(16, 8), (40, 24), (40, 40), (40, 100), (60, 150), (50, 200),
                                 (40, 70), (90, 120)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("core", [0, 2, 3])
def test_rounding(n, r, bad, core):
    dims = [n] * 3 + ([n] if (n, r) in ((16, 8), (40, 24)) else [n - 5])
    z = O.gauss_tt(dims, [1] + [r] * 3 + [1], r, 0.1)
    tol = 1e-8 * O.norm(z)
    good = O.truncate(z, tol, z.r)
    cores = [c.copy() for c in z.cores]
    cores[core][cores[core].size // 3] = bad
    dz = P.DevTT.from_host(O.HostTT(z.n, z.r, cores))
    P.truncate(dz, tol, z.r)
    out = to_host(dz)
    assert out.r[0] == out.r[-1] == 1 and all(1 <= a <= b for a, b in zip(out.r, z.r))
    assert not all(np.all(np.isfinite(c)) for c in out.cores)
    dz = P.DevTT.from_host(z)
    P.truncate(dz, tol, z.r)
    out = to_host(dz)
    assert out.r == good.r and O.rel_diff(out, good) < 1e-11


@pytest.mark.parametrize("r", [3, 16, 17, 40, 48, 64, 70])
@pytest.mark.parametrize("where", ["x", "y"])
@pytest.mark.parametrize("core", [1, 2])
def test_inner_product_of_positive_trains_with_an_infinity(r, where, core):
    """Every other term is positive: the sum is infinite and not NaN."""
    rng = np.random.default_rng(r)
    n, ranks = [20, 70, 33, 9], [1, r, max(1, r - 2), r, 1]
    t = {q: O.HostTT(n, ranks, [rng.random(ranks[k] * n[k] * ranks[k + 1]) + 0.1
                                for k in range(4)]) for q in "xy"}
    t[where].cores[core][-7] = np.inf
    assert P.dotprod(P.DevTT.from_host(t["x"]), P.DevTT.from_host(t["y"])) == np.inf
