"""Roundings of large cores whose left unfoldings have conditions between 4 and 30: one
Cholesky-QR pass, and Q = A T formed on the second stream from the place where the
rounding keeps T.  The same bits as without that stream, and the oracle's result."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from gpu_util import to_host

pytestmark = pytest.mark.gpu


def _train(n, r, d, s, seed):
    """Gaussian cores whose left unfoldings' columns share one more Gaussian column
    times s (condition some sqrt(1 + r s^2))."""
    x = O.gauss_tt([n] * d, [1] + [r] * (d - 1) + [1], seed, 0.05)
    rng = np.random.default_rng(seed)
    cores = []
    for k, c in enumerate(x.cores):
        u = c.reshape(-1, x.r[k + 1], order="F").copy()
        if k < d - 1:
            u += 0.05 * s * rng.standard_normal((u.shape[0], 1))
        cores.append(u.ravel(order="F"))
    return O.HostTT(x.n, x.r, cores)


@pytest.mark.parametrize("r,cap,mixed", [(128, 64, False), (100, 100, False), (128, 64, True)])
def test_side_stream_bitwise_equal(r, cap, mixed):
    n, d = 512, 5
    z = _train(n, r, d, 0.6, r)
    caps = [1] + [cap] * (d - 1) + [1]
    tol = 1e-8 * O.norm(z)
    L = P.lib()
    L.ptt_hip_side_enabled.restype = C.c_int
    L.ptt_hip_side_enable.argtypes = [C.c_int]
    was = L.ptt_hip_side_enabled()
    outs = []
    P.set_leaf_precision(1 if mixed else 0)
    try:
        for on in (1, 0, 1):
            L.ptt_hip_side_enable(on)
            dz = P.DevTT.from_host(z)
            P.truncate(dz, tol, caps)
            st = P.last_round_stats()
            outs.append(to_host(dz))
            dz.free()
            for k in range(1, d - 1):
                assert 4.0 < st.kappa_ltr[k] <= 30.0
                assert st.ltr_cholqr_passes[k] == (2 if mixed else 1)
    finally:
        L.ptt_hip_side_enable(was)
        P.set_leaf_precision(0)
    for o in outs[1:]:
        assert o.r == outs[0].r
        for a, b in zip(o.cores, outs[0].cores):
            np.testing.assert_array_equal(a, b)
    ref = O.truncate(z, tol, caps)
    assert outs[0].r == ref.r
    # beside a cut between nearly tied singular values
    assert O.rel_diff(outs[0], ref) < 1e-10
