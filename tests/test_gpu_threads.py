"""Calls that share no train and no scratch memory, from several threads at once:
formal sums in all of them, and beside those one thread whose calls upload
coefficients.  Against the same calls from one thread, bit for bit."""
import threading

import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P
from gpu_util import to_host

pytestmark = pytest.mark.gpu


def _run(jobs):
    err = []

    def call(f):
        try:
            f()
        except BaseException as e:  # noqa: BLE001
            err.append(e)

    ts = [threading.Thread(target=call, args=(f,)) for f in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not err, err


def _sums(i, out, reps):
    n = [7, 8, 9, 10]
    x = O.gauss_tt(n, [1, 3, 4 + i, 2, 1], 10 + i)
    y = O.gauss_tt(n, [1, 2, 2, 5, 1], 50 + i)
    dx, dy = P.DevTT.from_host(x), P.DevTT.from_host(y)
    ref = O.axpby(2.0, x, -1.0, y)

    def job():
        for _ in range(reps):
            out[i] = P.axpby(2.0, dx, -1.0, dy)
    return job, ref


def _same(dev, ref):
    got = to_host(dev)
    assert got.r == ref.r
    for a, b in zip(got.cores, ref.cores):
        np.testing.assert_array_equal(a, b)


def test_formal_sums():
    out = {}
    jobs = [_sums(i, out, 400) for i in range(8)]
    _run([j for j, _ in jobs])
    for i, (_, ref) in enumerate(jobs):
        _same(out[i], ref)


def test_uploads_beside_formal_sums():
    rng = np.random.default_rng(3)
    n, reps = 64, 300
    coef = rng.standard_normal((reps, n)) * 0.01 + 1.0
    x = O.gauss_tt([n] * 3, [1, 5, 5, 1], 9)
    L = P.lib()

    def scaled(dev):
        def job():
            for c in coef:
                P_, p = P._dp(c)
                L.attac_mult_diag_mat(dev.tt, 1, p)
        return job

    one, many = P.DevTT.from_host(x), P.DevTT.from_host(x)
    scaled(one)()
    out = {}
    jobs = [_sums(i, out, 300) for i in range(6)]
    _run([j for j, _ in jobs] + [scaled(many)])
    _same(many, to_host(one))
    for i, (_, ref) in enumerate(jobs):
        _same(out[i], ref)
