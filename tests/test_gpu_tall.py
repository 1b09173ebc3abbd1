"""Roundings whose last bond has more rows than columns (mode size below the formal
rank), against the oracle: columns on either side of where the SVD starts from the
small Gram's vectors (32, 192) and of its kernels' sizes, cut by the cap, by the
tolerance and not at all, with a rank-deficient last core."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P

pytestmark = pytest.mark.gpu


def _check(z, tol, caps, bar):
    ref = O.truncate(z, tol, caps)
    dz = P.DevTT.from_host(z)
    P.truncate(dz, tol, caps)
    out = O.HostTT(dz.n, dz.r, dz.download_cores())
    assert out.r == ref.r
    assert O.rel_diff(out, ref) < bar


@pytest.mark.parametrize("last,rx,ry", [(32, 25, 15), (33, 20, 15), (48, 40, 30), (64, 60, 40),
                                        (65, 40, 30), (96, 70, 60), (129, 80, 70), (192, 110, 100),
                                        (193, 110, 100)])
@pytest.mark.parametrize("cut", ["none", "cap"])
def test_sum(last, rx, ry, cut):
    n = [30, 40, last]
    x = O.gauss_tt(n, [1, rx, rx, 1], 1, 0.2)
    y = O.gauss_tt(n, [1, ry, ry, 1], 2, 0.2)
    z = O.axpby(1.0, x, 1.0, y)
    caps = list(z.r) if cut == "none" else [1, 20, max(rx, ry) // 2, 1]
    # 1e-12 of the norm beside a cut between nearly tied singular values
    _check(z, 1e-10 * O.norm(z), caps, 1e-11)


def test_update_and_deficient_core():
    n = [30, 40, 50]
    x = O.gauss_tt(n, [1, 40, 40, 1], 1, 0.2)
    y = O.gauss_tt(n, [1, 30, 30, 1], 2, 0.2)
    z = O.axpby(1.0, x, 1e-10, y)
    _check(z, 1e-8 * O.norm(z), list(z.r), 1e-7)
    c = [a.copy() for a in z.cores]
    last = c[2].reshape(70, 50, order="F")
    last[:, 25:] = last[:, :25]
    c[2] = last.ravel(order="F")
    w = O.HostTT(z.n, z.r, c)
    _check(w, 1e-8 * O.norm(w), list(w.r), 1e-7)
