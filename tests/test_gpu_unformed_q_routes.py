"""Which way the roundings of test_gpu_unformed_q take, from their statistics: one pass
and a condition up to 4 (Q left unformed) before an ill-conditioned core, several passes
or the change-over to the Householder trees at it."""
import pytest

import oracle_lib as O
import paratt_amd as P
from test_gpu_unformed_q import _train

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [20, 32, 40, 100, 128])
@pytest.mark.parametrize("bad", [None, 1, 3])
def test_conditions_and_passes(r, bad):
    z = _train([200, 90, 90, 90, 140], r, bad, r)
    dz = P.DevTT.from_host(z)
    P.truncate(dz, 1e-10 * O.norm(z), [1] + [r] * 4 + [1])
    st = P.last_round_stats()
    passes, kappa = list(st.ltr_cholqr_passes[:4]), list(st.kappa_ltr[:4])
    first = 4 if bad is None else bad
    assert passes[:first] == [1] * first
    # (core 0 has no more than 200 rows: its condition is that of a nearly square one)
    assert all(1.0 <= k <= 4.0 for k in kappa[1:first]) and 1.0 <= kappa[0] <= 30.0
    if bad is not None and r <= 32:
        assert passes[bad:] == [0] * (4 - bad)
    elif bad is not None:
        assert passes[bad] > 1 and kappa[bad] > 1e3
