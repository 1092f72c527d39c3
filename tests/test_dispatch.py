"""The operators' choice of kernel, on the CPU.

Which forms a call may take where its result lies in the memory of its
operands: a work-group of a one-launch form writes while others still read, so
these calls take forms that read everything first.  And g2_matmul's forms under
graph capture, which share no buffer.  No GPU is involved, the addresses are
numbers."""
import ctypes as C
import random

import pytest

import g2hip

lib = C.CDLL(g2hip.LIB_PATH)
F = 4


@pytest.mark.parametrize("NH,S,T", [(1, 256, 256), (2, 1024, 1), (12, 1024, 200), (25, 700, 256)])
def test_attention_in_one_launch_reads_what_it_does_not_write(NH, S, T):
    fn = lib.g2i_attn_one_launch
    fn.argtypes = [C.c_void_p] * 4 + [C.c_int] * 3
    D = 64 * NH
    q, k, v, out = 1 << 20, 1 << 24, 1 << 28, 1 << 30
    kend, vend = k + ((D - 1) * S + T) * F, v + T * D * F
    assert fn(q, k, v, out, T, D, S) == 1
    assert fn(q, k, v, out, 257, D, S) == 0 and fn(q, k, v, out, 0, D, S) == 0  # too long; a length on the device
    assert fn(q, k, v, q, T, D, S) == 1  # each head's queries, by the work-group that has read them
    for o in (q + F, q - F, q + 64 * F, q + (D - 1) * F, q - (D - 1) * F):
        assert fn(q, k, v, o, T, D, S) == (1 if D == 64 and abs(o - q) >= 64 * F else 0)
    for o in (q + D * F, q - D * F, k - D * F, kend, v - D * F, vend):  # beside them
        assert fn(q, k, v, o, T, D, S) == 1
    for o in (k, k - (D - 1) * F, kend - F, v, v - (D - 1) * F, vend - F):
        assert fn(q, k, v, o, T, D, S) == 0


def test_attention_output_over_its_operands():
    fn = lib.g2i_attn_out_groups
    fn.argtypes = [C.c_void_p] * 3 + [C.c_int] * 3
    scores, v = 1 << 24, 1 << 28
    for D, DH, T in ((64, 64, 300), (48, 16, 7), (10, 1, 1)):
        for base, size in ((scores, ((D - 1) // DH * 1024 + T) * F), (v, T * D * F)):
            for at, groups in ((0, 4), (size - F, 4), (size, 1), (F - D * F, 4), (-D * F, 1)):
                assert fn(scores, v, base + at, T, D, DH) == groups


@pytest.mark.parametrize("b_size", [4, 2])
@pytest.mark.parametrize("N,K", [(1, 1), (64, 300), (700, 20)])
def test_matvec_over_its_operands(N, K, b_size):
    fn = lib.g2i_matvec_apart
    fn.argtypes = [C.c_void_p] * 2 + [C.c_size_t] + [C.c_void_p] * 3 + [C.c_int] * 2
    A, B, bias, res = 1 << 24, 1 << 28, 1 << 30, 1 << 31
    for base, size in ((A, K * F), (B, N * K * b_size), (bias, N * F), (res, N * F)):
        for at in (0, size - b_size, F - N * F, size, -N * F):
            apart = at in (size, -N * F) or (at == 0 and base in (bias, res))
            assert fn(A, B, b_size, bias, res, base + at, N, K) == apart
            if base in (bias, res):
                assert fn(A, B, b_size, None, None, base + at, N, K) == 1


def matmul_pick(M, N, K, whole=False, cus=256):
    fn = lib.g2i_matmul_pick
    fn.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.POINTER(C.c_int)]
    splits = C.c_int()
    return fn(cus, M, N, K, whole, C.byref(splits)), splits.value


def test_captured_matmul_has_no_splits():
    rng = random.Random(7)
    split = 0
    for _ in range(3000):
        M, N, K = (int(2 ** rng.uniform(0, e)) for e in (10, 16, 14))
        split += matmul_pick(M, N, K)[1] > 1
        assert matmul_pick(M, N, K, whole=True)[1] == 1
        form, ks = matmul_pick(M, N, K)
        if ks == 1:  # without splits both choose alike
            assert matmul_pick(M, N, K, whole=True) == (form, 1)
    assert split > 100


@pytest.mark.parametrize("b_size", [4, 2])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (64, 64, 64), (300, 48, 48), (10, 2000, 700)])
def test_matmul_over_its_operands(M, N, K, b_size):
    fn = lib.g2i_matmul_in_place
    fn.argtypes = [C.c_void_p] * 2 + [C.c_size_t, C.c_void_p] + [C.c_long] * 3
    A, B = 1 << 30, 1 << 32
    for base, size in ((A, M * K * F), (B, K * N * b_size)):
        for at, over in ((0, 1), (size - b_size, 1), (size, 0), (F - M * N * F, 1), (-M * N * F, 0)):
            assert fn(A, B, b_size, base + at, M, N, K) == over


def test_matmul_launches_stay_below_the_thread_limit():
    """Sizes up to all of the memory: at most g2i_matmul_rows rows a call, in a
    form whose launch has fewer than 2^32 threads."""
    rows = lib.g2i_matmul_rows
    rows.argtypes, rows.restype = [C.c_long], C.c_long
    tile = [(16, 32, 512), (32, 32, 512), (64, 64, 256), (128, 128, 256), (128, 128, 512)]
    rng = random.Random(3)
    narrowed = 0
    for _ in range(20000):
        N, K = (int(2 ** rng.uniform(0, e)) for e in (30, 12))
        if 2 * N * K > 2 ** 38 or rows(N) < 1:
            continue
        M = min(int(2 ** rng.uniform(0, 30)), max(1, 2 ** 36 // N))
        narrowed += M > rows(N)
        M = min(M, rows(N))
        form, ks = matmul_pick(M, N, K)
        bm, bn, threads = tile[form]
        assert -(-M // bm) * -(-N // bn) * threads < 2 ** 32, (M, N, K, form)
    assert narrowed > 10
    assert rows(2 ** 30 - 64) == 64 and rows(2 ** 30) == 0


FORMS = {0: (16, "direct, 16 rows"), 1: (32, "direct, 32 rows"), 2: (64, "64 x 64"), 3: (128, "128 x 128"),
         4: (128, "alternating groups")}


def test_matmul_tests_reach_every_form_on_ragged_sizes():
    """Each form of g2_matmul, whole and (64 x 64, alternating) in K splits, is
    chosen by a tested size that divides neither its rows nor its step of 32
    and has an odd number of columns, or, for the values' tests, some edge."""
    from test_matmul_gpu import EDGES, FORM_SIZES

    every = {(f, s) for f in FORMS for s in (False, True)} - {(0, True), (1, True), (3, True)}

    def reached(sizes, ragged):
        got = set()
        for M, N, K in sizes:
            form, ks = matmul_pick(M, N, K)
            if not ragged or (M % FORMS[form][0] and K % 32 and N % 2):
                got.add((form, ks > 1))
        return got

    assert reached(FORM_SIZES, False) == every
    assert reached(EDGES, True) | {(2, True)} == every  # splits of 64 x 64: an even 300 columns, 5007 = 156 * 32 + 15
    assert (2, True) in reached([s for s in EDGES if s[0] % 64 and s[2] % 32], False)


def matvec_form(f16, N, K, cus=256):
    slices = C.c_int()
    return lib.g2i_matvec_form(cus, int(f16), N, K, C.byref(slices)), slices.value


def test_matvec_forms():
    """The lanes and slices that the large matrices' test is there for, no
    choice outside the kernels and the scratch (eight slices of 65536), and no
    work-groups of a second round for a fifth of the chip: 10000 x 6400 fp16
    had 313 of them on 256 CUs."""
    from test_matvec_gpu import LARGE

    assert {matvec_form(*c)[0] for c in LARGE} == {8, 16, 64}
    assert {matvec_form(*c)[1] > 1 for c in LARGE if matvec_form(*c)[0] == 16} == {True}
    rng = random.Random(11)
    for _ in range(5000):
        f16, N, K = rng.random() < 0.5, int(2 ** rng.uniform(0, 16)), int(2 ** rng.uniform(0, 14))
        lanes, slices = matvec_form(f16, N, K)
        assert lanes in ((4, 8, 16) if f16 else (4, 8, 16, 64)) and 1 <= slices <= 8 and slices <= K
    for f16, N, K in ((True, 10000, 6400), (False, 10000, 6400), (False, 20000, 6400), (False, 25000, 4096)):
        lanes, slices = matvec_form(f16, N, K)
        rounds = -(-N // (lanes * (8 if f16 else 4))) * slices / 256
        assert rounds / -(-rounds // 1) > 0.75
