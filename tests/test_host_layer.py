"""What the C host layer queues and allocates, on a CPU: its sources compiled
against host_stub.c, which stands in for the kernels without computing anything."""
import ctypes as C
import os
import subprocess

import pytest

import paratt_amd as P

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "paratt_amd", "csrc", "host")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host.so")
    subprocess.run(["gcc", "-std=c99", "-O1", "-fPIC", "-shared", "-DPARATT_AMD_NO_MPI",
                    "-I" + os.path.join(ROOT, "include"), "-I" + HOST,
                    os.path.join(ROOT, "tests", "host_stub.c"), os.path.join(HOST, "round.c"),
                    os.path.join(HOST, "tt.c"), "-o", so, "-lm"], check=True, timeout=120)
    L = C.CDLL(so)
    PP, IP = C.POINTER(P.Paratt), C.POINTER(C.c_int)
    L.alloc_ptt.restype = PP
    L.free_ptt.argtypes = [PP]
    L.alloc_tt.restype = C.POINTER(P.AttacTT)
    L.free_tt.argtypes = [C.POINTER(P.AttacTT)]
    L.rank_change_tt.argtypes = [C.POINTER(P.AttacTT), IP]
    L.paratt_amd_truncate_rel.argtypes = [PP, C.c_double, IP]
    L.paratt_amd_truncate_rel_sketch.argtypes = [PP, C.c_double, IP, IP]
    L.paratt_amd_last_sketch_counts.argtypes = [IP]
    return L


def _ints(v):
    return (C.c_int * len(v))(*v)


def _count(L, name):
    return C.c_long.in_dll(L, name).value


def _set_condition(L, kappa, deficient=0):
    C.c_double.in_dll(L, "stub_kappa").value = kappa
    C.c_int.in_dll(L, "stub_deficient").value = deficient


@pytest.mark.parametrize("kappa,side,main", [(1.5, 0, 0), (4.0, 0, 0), (4.1, 2, 1), (30.0, 2, 1)])
def test_formed_q_of_a_rounding_goes_to_the_side_stream(lib, kappa, side, main):
    """One-pass bonds: left unformed up to a condition of 4; beyond it the products of
    cores of at least 4M elements (the middle two) run on the side stream."""
    n, r = [300] * 4, [1, 128, 128, 128, 1]
    x = lib.alloc_ptt(4, _ints(n), _ints(r))
    _set_condition(lib, kappa)
    lib.stub_reset()
    lib.paratt_amd_truncate_rel(x, 1e-8, _ints([1, 64, 64, 64, 1]))
    assert list(x.contents.x.contents.ttRank[:5]) == [1, 64, 64, 64, 1]
    got = (_count(lib, "stub_side_inplace"), _count(lib, "stub_main_inplace"))
    lib.free_ptt(x)
    assert got == (side, main)


def _queued(L):
    return tuple(_count(L, "stub_" + k) for k in ("chol", "tree_factors", "eigen", "mallocs"))


# every bond at most 16 columns: trees; 24 columns: Gram route while well conditioned,
# trees behind the first core that is not; 40: Gram route
@pytest.mark.parametrize("r,kappa,pred", [
    (r, kappa, pred) for r, kappa in ((10, 1.5), (16, 1e7), (24, 1.5), (24, 1e7), (40, 1.5))
    for pred in (0, 13, 200, None)])
def test_rounding_without_a_usable_prediction_is_the_plain_one(lib, r, kappa, pred):
    """A sketch takes at least 9 columns and at most half of the bond's and 128."""
    n, ranks = [50] * 5, [1, r, r, r, r, 1]
    mr = _ints([1] + [5] * 4 + [1])
    _set_condition(lib, kappa)
    got = []
    for sketch in (0, 0, 1):  # the first one grows the scratch memory
        x = lib.alloc_ptt(5, _ints(n), _ints(ranks))
        lib.stub_reset()
        if sketch:
            p = None if pred is None else _ints([0] + [pred] * 4 + [0])
            lib.paratt_amd_truncate_rel_sketch(x, 1e-8, mr, p)
        else:
            lib.paratt_amd_truncate_rel(x, 1e-8, mr)
        got.append(_queued(lib))
        lib.free_ptt(x)
    assert got[2] == got[1]
    cnt = (C.c_int * 2)()
    lib.paratt_amd_last_sketch_counts(cnt)
    assert list(cnt) == [0, 0]


@pytest.mark.parametrize("kappa,trees", [(1.5, 0), (1e7, 3)])
def test_refused_predictions_round_again_only_where_the_trees_would(lib, kappa, trees):
    """24 columns, sketches of 12 that the stub's residual refuses: at most one
    eigensolver call a bond."""
    x = lib.alloc_ptt(5, _ints([50] * 5), _ints([1, 24, 24, 24, 24, 1]))
    _set_condition(lib, kappa)
    lib.stub_reset()
    lib.paratt_amd_truncate_rel_sketch(x, 1e-8, _ints([1] + [5] * 4 + [1]),
                                       _ints([0, 4, 4, 4, 4, 0]))
    cnt = (C.c_int * 2)()
    lib.paratt_amd_last_sketch_counts(cnt)
    eigen, factors = _count(lib, "stub_eigen"), _count(lib, "stub_tree_factors")
    lib.free_ptt(x)
    assert list(cnt) == [4, 0]
    assert eigen <= 4 and factors == trees


def test_growing_a_train_waits_once_and_keeps_little_of_the_old(lib):
    """Small trains free all of their old cores at once; a large one never holds more
    than 1 GiB and one core of them besides its new ones."""
    for n, r, grown in ((20, 10, 12), (1000, 280, 400)):
        x = lib.alloc_tt(9, _ints([n] * 9), _ints([1] + [r] * 8 + [1]))
        lib.stub_reset()
        lib.rank_change_tt(x, _ints([1] + [grown] * 8 + [1]))
        live = C.c_size_t.in_dll(lib, "stub_live").value
        peak = C.c_size_t.in_dll(lib, "stub_peak").value
        frees = _count(lib, "stub_frees")
        lib.free_tt(x)
        assert peak - live <= 2 ** 30 + 8 * n * r * r
        assert frees == 1 if n == 20 else frees <= 6


@pytest.mark.parametrize("bad", [1, 2, 3])
def test_unformed_qs_are_formed_where_the_trees_take_over(lib, bad):
    """24 columns: the cores before the first ill-conditioned one after core 0 hold A
    with Q unformed; the trees take over there and get every one of those Qs."""
    x = lib.alloc_ptt(5, _ints([50] * 5), _ints([1, 24, 24, 24, 24, 1]))
    _set_condition(lib, 1.5)
    lib.stub_reset()
    C.c_long.in_dll(lib, "stub_bad_chol").value = bad
    lib.paratt_amd_truncate_rel(x, 1e-8, _ints([1] + [5] * 4 + [1]))
    C.c_long.in_dll(lib, "stub_bad_chol").value = -1
    got = tuple(_count(lib, "stub_" + k) for k in ("chol", "main_inplace", "side_inplace",
                                                   "tree_factors"))
    lib.free_ptt(x)
    assert got == (bad + 1, bad, 0, 4 - bad)


@pytest.mark.parametrize("n,r,trees", [(50, 16, True), (511, 16, True), (512, 16, False),
                                       (745, 11, False), (744, 11, True), (4096, 10, True),
                                       (4096, 16, False), (50, 17, False)])
def test_trains_that_the_trees_take_from_the_start(lib, n, r, trees):
    """Up to 16 columns, but not 11 to 16 with 8192 rows or more."""
    x = lib.alloc_ptt(5, _ints([n] * 5), _ints([1] + [r] * 4 + [1]))
    _set_condition(lib, 1.5)
    lib.stub_reset()
    lib.paratt_amd_truncate_rel(x, 1e-8, _ints([1] + [5] * 4 + [1]))
    got = (_count(lib, "stub_tree_factors"), _count(lib, "stub_chol") > 0)
    lib.free_ptt(x)
    assert got == ((4, False) if trees else (0, True))
