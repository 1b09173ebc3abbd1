"""Roundings that leave Q = A T unformed on the way right: well-conditioned bonds
beside ill-conditioned ones (whose Q is formed), and trains of 17 to 32 columns that
change over to the Householder trees behind cores whose Q is still unformed.  Against
the oracle; the bar is the other roundings' where a cut meets nearly tied values."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P

pytestmark = pytest.mark.gpu


def _train(n, r, bad, seed):
    """Gaussian cores; core `bad` has half of its left unfolding's columns within 1e-6 of
    the others (condition of its factor some 1e6)."""
    d = len(n)
    x = O.gauss_tt(n, [1] + [r] * (d - 1) + [1], seed, 0.3)
    cores = [c.copy() for c in x.cores]
    if bad is not None:
        u = cores[bad].reshape(-1, r, order="F")
        h = r // 2
        u[:, h:2 * h] = u[:, :h] + 1e-6 * u[:, h:2 * h]
        cores[bad] = u.ravel(order="F")
    return O.HostTT(x.n, x.r, cores)


@pytest.mark.parametrize("r", [20, 32, 40, 100, 128])
@pytest.mark.parametrize("bad", [None, 1, 3])
@pytest.mark.parametrize("cap", [0, 11])
def test_matches_oracle(r, bad, cap):
    n = [200, 90, 90, 90, 140]
    z = _train(n, r, bad, r)
    caps = [1] + [cap or r] * 4 + [1]
    tol = 1e-10 * O.norm(z)
    ref = O.truncate(z, tol, caps)
    dz = P.DevTT.from_host(z)
    P.truncate(dz, tol, caps)
    out = O.HostTT(dz.n, dz.r, dz.download_cores())
    assert out.r == ref.r
    assert O.rel_diff(out, ref) < 1e-11
