"""g2_matmul's forms at the sizes where they can go wrong, the values that
bf16 parts cannot carry and the accuracy that the parts are there for, against
the CPU oracle's fp32 product and against 64 bits.

The sizes put each form (direct 16- and 32-row tiles, 64x64 tiles whole and in
K splits, 128x128 tiles of several work-groups per CU, and of alternating wave
groups whole and in K splits) on ragged edges: one row or column past a tile,
odd column counts (a column pair that the last column begins), K below one
step of 32, one past it, and splits that end in a partial step.  That they do
is checked against the choice itself in test_dispatch.py.
"""
import ctypes as C
import time

import numpy as np
import pytest

from oracle import oracle
from parity import assert_close_bound, dot_bound

pytestmark = pytest.mark.gpu


def operands(M, N, K, f16, seed):
    r = np.random.default_rng(seed)
    A = r.standard_normal((M, K)).astype(np.float32)
    B = (0.02 * r.standard_normal((K, N))).astype(np.float32)
    if f16:
        B = B.astype(np.float16).astype(np.float32)
    return A, B, r.standard_normal(N).astype(np.float32)


def product(g2, A, B, bias, f16):
    (M, K), N = A.shape, B.shape[1]
    dC = g2.to_device(np.full(M * N + 64, 7.0, np.float32))
    dB = g2.to_device(g2.convert_f16(B) if f16 else B)
    g2.matmul(g2.to_device(A), dB, None if bias is None else g2.to_device(bias), dC, M, N, K, f16=f16)
    got = dC.download(np.float32, M * N + 64)
    assert (got[M * N:] == 7.0).all()  # nothing past the matrix
    return got[:M * N].reshape(M, N)


EDGES = [
    (1, 1, 1), (1, 1, 40), (17, 1, 65), (3, 2, 31),            # 64 x 64; one column: no pairs
    (16, 31, 32), (333, 1601, 96), (470, 2305, 70), (641, 12801, 32),  # 64 x 64
    (40, 300, 5007),                                           # 64 x 64 in 12 splits
    (17, 33, 33), (15, 65, 257), (33, 97, 300), (65, 129, 1000), (130, 257, 2049),  # direct, 16 rows
    (50, 3203, 259), (18, 5755, 1389),                         # direct, 32 rows
    (700, 8321, 70), (657, 12803, 40),                         # 128 x 128
    (118, 20173, 1191), (200, 9001, 300),                      # 128 x 128, alternating groups
    (257, 5121, 1281),                                         # alternating groups in 2 splits
]


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("M,N,K", EDGES)
def test_matmul_edges(g2, M, N, K, f16):
    A, B, bias = operands(M, N, K, f16, M + N + K)
    bound = dot_bound(np.abs(A).astype(np.float64), np.abs(B).astype(np.float64), K)
    assert_close_bound(product(g2, A, B, bias, f16), oracle.matmul(A, B, bias, M, N, K), bound, what="matmul")
    assert_close_bound(product(g2, A, B, None, f16), oracle.matmul(A, B, None, M, N, K), bound, what="no bias")


# a ragged size per form: direct 16 and 32 rows, 64x64 whole and split, 128x128 of
# several work-groups per CU, of alternating wave groups whole and split
FORM_SIZES = [(20, 70, 100), (18, 5755, 1389), (470, 2305, 70), (70, 200, 4100), (700, 8321, 70), (118, 20173, 1191),
              (257, 5121, 1281)]


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("M,N,K", FORM_SIZES)
def test_matmul_special_values(g2, M, N, K, f16):
    """Rows with an infinity, a NaN, a value that rounds past bf16's largest,
    and rows of magnitudes whose low parts bf16 cannot hold."""
    A, B, _ = operands(M, N, K, f16, 5)
    A[1, 7], A[2, 9], A[3, 11], A[M - 1, K - 1] = np.inf, np.nan, -np.inf, np.inf
    A[4] *= np.float32(2.0) ** -112
    A[5] = 0
    A[6], A[7] = 0, 0
    A[6, 3], A[7, K - 1] = 3.4e38, -3.4e38
    B[:, 2] = 0.5
    with np.errstate(all="ignore"):
        ref = oracle.matmul(A, B, None, M, N, K)
        got = product(g2, A, B, None, f16)
        bound = dot_bound(np.abs(A).astype(np.float64), np.abs(B).astype(np.float64), K)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    fin = np.isfinite(ref)
    np.testing.assert_array_equal(got[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
    assert (np.abs(got[fin].astype(np.float64) - ref[fin]) <= bound[fin] + 1e-45).all()


def sum_bound(K):
    """What the norm of K random terms' fp32 sum may be off by, of its own: a
    product's left-out parts are 2^-24 of it at most, and the sum takes about
    K / 5 roundings (six instructions per 32 k) of at most 2^-24 of a partial
    sum that grows to its own size, which add up to some sqrt(K / 15) of them.
    Measured 0.5 to 5 times 2^-24 for K 70 to 4100; without the third parts
    it is 57 times (test_matmul_bound.py)."""
    return 2.0 ** -24 * (3 + np.sqrt(K) / 3)


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("M,N,K", FORM_SIZES)
def test_matmul_accuracy(g2, M, N, K, f16):
    """Every row's and every column's error, in the norm, against 64 bits."""
    r = np.random.default_rng(M)
    A, B = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    if f16:
        B = B.astype(np.float16).astype(np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    err = product(g2, A, B, None, f16) - ref
    for axis in (0, 1):
        assert (np.linalg.norm(err, axis=axis) <= sum_bound(K) * np.linalg.norm(ref, axis=axis)).all()


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("M,N,K", FORM_SIZES)
def test_matmul_low_parts(g2, M, N, K, f16):
    """Results that rest on the second and third parts: a row of A or a column
    of B that picks one row or column of the other is that one, every bit; a
    row of pairs whose products cancel but for 2^-12; factors whose left-out
    products are the largest."""
    r = np.random.default_rng(N)
    A, B = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    A[1], B[:, 1] = 0, 0
    A[1, K - 1], B[K - 3, 1] = 1, 1
    H = K // 2
    A[2, H:2 * H] = A[2, :H]
    B[H:2 * H, 5] = -B[:H, 5] * np.float32(1 + 2.0 ** -12)
    A[3], B[:, 4] = 1 + 2.0 ** -8 - 2.0 ** -17, 1 + 2.0 ** -8 - 2.0 ** -17
    if f16:
        B = B.astype(np.float16).astype(np.float32)
    got = product(g2, A, B, None, f16)
    np.testing.assert_array_equal(got[1], B[K - 1])
    np.testing.assert_array_equal(got[:, 1], A[:, K - 3])
    exact = A.astype(np.float64) @ B.astype(np.float64)
    terms = np.linalg.norm(A[2].astype(np.float64) * B[:, 5])
    assert abs(got[2, 5] - exact[2, 5]) <= 4 * sum_bound(K) * terms  # one output: four deviations
    # K equal terms: a rounding of up to 2^-24 of the whole for each of K / 5 steps
    assert abs(got[3, 4] / exact[3, 4] - 1) <= 2.0 ** -24 * (2 + K / 10)


def sized(r, shape, e):
    """Values of magnitude 2^e to 2^(e+1), all 24 bits random."""
    return np.ldexp(np.float32(1) + r.random(shape, np.float32), e).astype(np.float32) * r.choice(np.float32([-1, 1]), shape)


@pytest.mark.parametrize("f16,ea,eb", [(False, -115, 70), (False, 70, -120), (False, -126, 100), (False, -140, 100),
                                       (True, -120, 10), (True, -140, 12)])
@pytest.mark.parametrize("M,N,K", FORM_SIZES)
def test_matmul_small_by_large(g2, M, N, K, f16, ea, eb):
    """Operands whose low bits bf16 parts do not hold, against ones that lift
    the product back among ordinary values: fp32 products all the same.  A sum
    of K random terms takes roundings of 2^-24 of a partial sum that grows to
    its own size, sqrt(K) / 3 of them in the norm; a result in fp32's
    subnormals is off by half their step besides."""
    r = np.random.default_rng(K)
    A, B = sized(r, (M, K), ea), sized(r, (K, N), eb)
    if f16:
        B = B.astype(np.float16).astype(np.float32)
    got, ref = product(g2, A, B, None, f16).astype(np.float64), A.astype(np.float64) @ B.astype(np.float64)
    err = np.linalg.norm(got - ref) - 2.0 ** -150 * np.sqrt(M * N)
    assert err <= 2.0 ** -24 * (2 + np.sqrt(K) / 2) * np.linalg.norm(ref)


@pytest.mark.parametrize("M,N,K", FORM_SIZES)
def test_matmul_one_small_value(g2, M, N, K):
    """One subnormal value in each operand, alone with a large factor: in a row
    and a column that the tile's other values do not share."""
    A, B, _ = operands(M, N, K, False, 3)
    A[M - 1], B[:, N - 1] = 0, 0
    A[M - 1, K - 1], B[K - 1, 0] = 2.0 ** -140, 2.0 ** 120
    A[0, 0], B[0, N - 1] = -(2.0 ** 120), 2.0 ** -145
    got = product(g2, A, B, None, False)
    assert got[M - 1, 0] == 2.0 ** -20 and got[0, N - 1] == -(2.0 ** -25)


@pytest.mark.parametrize("M,N,K", [(70, 200, 4100), (256, 1280, 1280), (512, 4000, 640), (1024, 8192, 1600)])
def test_matmul_time_by_values(g2, M, N, K):
    """Products of small size (1e-10 by 1e-10) take the ordinary time, and an
    infinity in every row or operands that only fp32 holds about the fp32
    instruction's: direct, 64x64 split, 128x128 (measured 1.0 and up to 5 times
    the ordinary time; 10 to 60 when each such output was summed by itself)."""
    A, B, _ = operands(M, N, K, False, 4)
    dA, dB, dC = g2.DevBuf(A.nbytes), g2.DevBuf(B.nbytes), g2.DevBuf(4 * M * N)

    def seconds(a, b):
        dA.upload(a)
        dB.upload(b)
        best = 1.0
        for _ in range(5):
            g2.matmul(dA, dB, None, dC, M, N, K)
            g2.sync()
            t = time.perf_counter()
            for _ in range(10):
                g2.matmul(dA, dB, None, dC, M, N, K)
            g2.sync()
            best = min(best, time.perf_counter() - t)
        return best

    plain = seconds(A, B)
    assert seconds(A * np.float32(1e-10), B * np.float32(5e-9)) < 2 * plain
    rows = A.copy()
    rows[:, K // 2] = np.inf
    assert seconds(rows, B) < 8 * plain
    assert seconds(A * np.float32(2.0 ** -125), B) < 8 * plain


@pytest.mark.parametrize("small", [False, True], ids=["ordinary", "recomputed"])
@pytest.mark.parametrize("M,N", [(1, 64), (5, 33), (64, 64), (300, 64), (2000, 17)])
def test_matmul_over_a(g2, M, N, small):
    """X = X W in place, W of at most 64 columns; also where tiles are
    computed again on the fp32 instruction."""
    A, B, bias = operands(M, N, N, False, 6)
    if small:
        A, B = A * np.float32(2.0 ** -120), B * np.float32(2.0 ** 120)
    dA = g2.to_device(A)
    g2.matmul(dA, g2.to_device(B), g2.to_device(bias), dA, M, N, N)
    bound = dot_bound(np.abs(A).astype(np.float64), np.abs(B).astype(np.float64), N)
    assert_close_bound(dA.download(np.float32, M * N).reshape(M, N), oracle.matmul(A, B, bias, M, N, N), bound, what="in place")


@pytest.mark.parametrize("M,N,K", [(70, 200, 4100), (257, 5121, 1281)])
def test_matmul_captured(g2, M, N, K):
    """Sizes whose eager call splits K through the library's buffer: a recorded
    call, replayed on a stream of its own beside eager split calls of other
    operands, gives the recorded product every time, and the eager calls
    theirs."""
    hip, vp = C.CDLL("libamdhip64.so"), C.c_void_p
    hip.hipStreamBeginCapture.argtypes = [vp, C.c_int]
    hip.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(vp), vp, vp, vp, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [vp, vp]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [vp]
    hip.hipStreamCreateWithFlags.argtypes = [C.POINTER(vp), C.c_uint]
    hip.hipStreamSynchronize.argtypes = hip.hipStreamDestroy.argtypes = [vp]
    sets, dev = [operands(M, N, K, False, s) for s in (1, 2)], []
    for A, B, bias in sets:
        dev.append((g2.to_device(A), g2.to_device(B), g2.to_device(bias), g2.DevBuf(4 * M * N)))
    refs = [(A.astype(np.float64) @ B.astype(np.float64) + bias) for A, B, bias in sets]
    stream, side, graph, exe = g2._lib.g2_stream(), vp(), vp(), vp()
    assert hip.hipStreamCreateWithFlags(C.byref(side), 1) == 0
    g2.sync()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # hipStreamCaptureModeThreadLocal
    g2.matmul(*dev[0], M, N, K)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0) == 0
    try:
        for rep in range(20):
            assert hip.hipGraphLaunch(exe, side) == 0
            for _ in range(3):
                g2.matmul(*dev[1], M, N, K)
            assert hip.hipStreamSynchronize(side) == 0
            g2.sync()
            for d, ref in zip(dev, refs):
                got = d[3].download(np.float32, M * N).reshape(M, N)
                assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref), f"replay {rep}"
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(side)


@pytest.mark.parametrize("P", [70, 300, 1000])
def test_prefill_small_weights_large_gain(g2, P):
    """The fp32 prefill's GEMMs (more than 64 rows: bf16 parts, split and whole)
    with q/k/v and MLP weights of 2^-128 behind LayerNorm gains of 2^122."""
    cfg = g2.make_config(2, 768, 12, vocab_size=1000)
    w = g2.synth_weights(cfg, 77)
    gain, part = np.float32(2.0 ** 122), np.float32(2.0 ** -122)
    for i, layer in enumerate(w["layers"]):
        layer = list(layer)
        for norm, mat in ((0, 2), (6, 8)):
            layer[norm] = (layer[norm] * gain).astype(np.float32)
            layer[mat] = (layer[mat] * part).astype(np.float32)
        w["layers"][i] = tuple(layer)
    ids = np.random.default_rng(P).integers(0, cfg.vocab_size, P).astype(np.int32)
    m = g2.Model.from_host(cfg, w, g2.F32, g2.PATH_FUSED)
    m.prefill(ids)
    om = oracle.Model(cfg, w)
    om.prefill(ids)
    np.testing.assert_allclose(m.logits(), om.logits(), rtol=0, atol=1e-4)
    om.close()
    m.free()
