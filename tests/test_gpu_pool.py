"""Device memory kept for reuse: which freed block a request takes, data in a block
taken again, the bound on what is kept, and giving it back."""
import ctypes as C

import numpy as np
import pytest

import paratt_amd as P

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib():
    L = P.lib()
    L.ptt_hip_init()
    L.ptt_hip_malloc.restype = C.c_void_p
    L.ptt_hip_malloc.argtypes = [C.c_size_t]
    L.ptt_hip_free.argtypes = [C.c_void_p]
    L.ptt_hip_free_many.argtypes = [C.c_int, C.POINTER(C.c_void_p)]
    L.ptt_hip_h2d.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t]
    L.ptt_hip_d2h.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t]
    L.ptt_hip_trim()
    yield L
    L.ptt_hip_trim()


def _free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    assert P.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


# sizes are rounded up to 512 bytes below 1 MiB and to 64 KiB above; a block serves
# requests it exceeds by at most a quarter and 4 KiB
@pytest.mark.parametrize("size,unit", [(1 << 16, 512), (10 << 20, 1 << 16)])
def test_what_a_freed_block_serves(lib, size, unit):
    most = size - 4096
    least = -(-(most * 4) // 5 // unit) * unit  # want + want / 4 + 4096 >= size
    while least + least // 4 + 4096 < size:
        least += unit
    for want, same in ((size, True), (size - 8, True), (least, True), (least - unit, False),
                       (size + 8, False)):
        p = lib.ptt_hip_malloc(size)
        lib.ptt_hip_free(p)
        q = lib.ptt_hip_malloc(want)
        assert (q == p) == same, want
        lib.ptt_hip_free(q)
        lib.ptt_hip_trim()


def test_data_in_a_block_taken_again(lib):
    rng = np.random.default_rng(1)
    for n in (1, 1000, 100003):
        for _ in range(3):
            a, b = rng.random(n), np.empty(n)
            p = lib.ptt_hip_malloc(a.nbytes)
            lib.ptt_hip_h2d(p, a.ctypes.data, a.nbytes)
            lib.ptt_hip_d2h(b.ctypes.data, p, a.nbytes)
            lib.ptt_hip_free(p)
            assert np.array_equal(a, b)


def test_what_is_kept_is_bounded_and_given_back(lib):
    gib = 1 << 30
    before = _free_bytes()
    p = (C.c_void_p * 6)(*[lib.ptt_hip_malloc(2 * gib + gib // 2) for _ in range(6)])
    lib.ptt_hip_free_many(6, p)
    kept = before - _free_bytes()
    assert 5 * gib <= kept <= 8 * gib + gib // 4
    q = lib.ptt_hip_malloc(5 * gib)  # more than half of the bound: never kept
    lib.ptt_hip_free(q)
    assert before - _free_bytes() <= kept + gib // 4
    lib.ptt_hip_trim()
    assert before - _free_bytes() <= gib // 4
