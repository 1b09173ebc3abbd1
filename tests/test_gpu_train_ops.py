"""The train-wide streaming kernels (formal sum, stencil sum) at the sizes
where a launch splits: more cores than one launch holds, trains that mix
even and odd ranks (paired and single accesses), modes of length 1, 2 and
odd.  Bit-exact against the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P

pytestmark = pytest.mark.gpu

TRAINS = [
    ([5, 6], [1, 3, 1], [1, 2, 1]),
    ([1, 2, 3], [1, 2, 2, 1], [1, 4, 2, 1]),
    ([6, 5, 8, 7], [1, 4, 6, 2, 1], [1, 2, 3, 8, 1]),
    ([3] * 35, [1] + [2, 3] * 17 + [1], [1] + [4, 1] * 17 + [1]),
    ([301, 64], [1, 33, 1], [1, 8, 1]),
]


@pytest.mark.parametrize("n,rx,ry", TRAINS)
def test_formal_sum_of_a_train(n, rx, ry):
    rx, ry = rx[:len(n)] + [1], ry[:len(n)] + [1]
    x, y = O.gauss_tt(n, rx, 3), O.gauss_tt(n, ry, 4)
    z = P.axpby(1.25, P.DevTT.from_host(x), -0.75, P.DevTT.from_host(y))
    ref = O.axpby(1.25, x, -0.75, y)
    assert z.r == ref.r
    for got, want in zip(z.download_cores(), ref.cores):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n,r,_", TRAINS)
def test_stencil_sum_of_a_train(n, r, _):
    L = P.lib()
    L.paratt_amd_mode_sum.argtypes = [C.POINTER(P.Paratt), C.POINTER(C.c_double),
                                      C.POINTER(P.Paratt)]
    x = O.gauss_tt(n, r[:len(n)] + [1], 12)
    st = np.array([-0.25, 0.1, 0.4])
    ref = O.mode_sum(x, st)
    u, s = P.DevTT.from_host(x), P.DevTT(x.n, [1] * (len(n) + 1))
    L.paratt_amd_mode_sum(u.p, st.ctypes.data_as(C.POINTER(C.c_double)), s.p)
    assert s.r == ref.r
    for got, want in zip(s.download_cores(), ref.cores):
        np.testing.assert_array_equal(got, want)
