"""Roundings of trains of at most 16 columns on either side of the rows from which they
start on the Cholesky-QR sweep: well-conditioned ones, which stay there, and formal sums
of a train with itself, which change over to the Householder trees.  Bars as of the
trees' other tests."""
import pytest

import oracle_lib as O
from test_gpu_tree import U, _round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,r", [(511, 16), (512, 16), (744, 11), (745, 11), (900, 10), (1100, 13)])
@pytest.mark.parametrize("same", [False, True])
@pytest.mark.parametrize("eps", [1e-8, 0.3])
def test_matches_oracle(n, r, same, eps):
    d = 5
    a, b = (r + 1) // 2, r // 2
    if same:
        a = b = r // 2
    x = O.gauss_tt([n] * d, [1] + [a] * (d - 1) + [1], 1, 0.05)
    y = x if same else O.gauss_tt([n] * d, [1] + [b] * (d - 1) + [1], 2, 0.05)
    z = O.axpby(1.0, x, 1e-3 if same else 1.0, y)
    ref = O.truncate(z, eps * O.norm(z), z.r)
    out, stats = _round(z, eps, z.r)
    assert out.r == ref.r
    # the cut at 0.3 leaves no more than the gap of a random train's singular values
    assert O.rel_diff(out, ref) < 64 * d * U * (1.0 if eps < 1e-3 else 1e5) + 1e-11
    tall = a + b > 10 and n * (a + b) >= 8192
    passes = list(stats.ltr_cholqr_passes[:d - 1])
    if not tall:
        assert max(passes) == 0
    elif not same:
        assert passes == [1] * (d - 1)
    else:
        assert max(passes[1:]) == 0
