"""Inner products against numpy at the edges of the one-mode kernel: ranks on either side
of its blocks of 16 and of its sizes (16, 32, 64), beyond it (65), ranks that differ between
the trains and along them, few and many mode indices.  The sums have positive terms, so
the tolerance is that of their roundings, (d + n r) u."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _positive(n, r, seed):
    rng = np.random.default_rng(seed)
    return [(rng.random((r[k], n[k], r[k + 1])) + 0.1) / r[k] for k in range(len(n))]


def _check(n, rx, ry, seed=1):
    xs, ys = _positive(n, rx, seed), _positive(n, ry, seed + 1)
    dx = P.DevTT.from_host(O.HostTT(n, rx, [c.ravel(order="F") for c in xs]))
    dy = P.DevTT.from_host(O.HostTT(n, ry, [c.ravel(order="F") for c in ys]))
    a = np.ones((1, 1))
    for x, y in zip(xs, ys):
        b = np.tensordot(a, x, axes=(0, 0))                          # (ry0, n, rx1)
        a = np.tensordot(b, y, axes=((0, 1), (0, 1))) / y.shape[1]   # (rx1, ry1)
    got, ref = P.dotprod(dx, dy), float(a[0, 0])
    tol = sum(n[k] + rx[k] + ry[k] + 4 for k in range(len(n))) * U
    assert abs(got - ref) <= tol * abs(ref), (got, ref)


@pytest.mark.parametrize("r", [1, 2, 3, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65])
@pytest.mark.parametrize("n", [1, 5, 33, 300])
def test_equal_ranks(r, n):
    _check([n, n, n + 1, n], [1, r, r, r, 1], [1, r, r, r, 1])


@pytest.mark.parametrize("rx,ry", [((1, 64, 3, 20, 1), (1, 5, 64, 1, 1)),
                                   ((1, 17, 16, 33, 1), (1, 1, 50, 2, 1)),
                                   ((1, 70, 12, 64, 1), (1, 9, 80, 31, 1))])
def test_unequal_ranks(rx, ry):
    _check([40, 7, 513, 64], list(rx), list(ry))


def test_many_indices_a_workgroup():
    _check([20, 1100, 1025, 9000, 3], [1, 20, 64, 40, 6, 1], [1, 30, 33, 64, 7, 1])
