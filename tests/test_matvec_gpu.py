"""g2_matvec and g2_matvec_sk at the sizes where their launches can go wrong:
rows shorter than one 16-byte vector, columns past the last whole vector or
column group, K below and above the rows that a work-group takes at once, the
column-lane choices, the sliced forms of tall narrow and of large matrices, operands at odd
addresses and results that overlap an operand; and the elementwise operators'
and the LayerNorm's remainders; against the CPU oracle."""
import numpy as np
import pytest

from oracle import oracle
from parity import assert_close_bound, dot_bound

pytestmark = pytest.mark.gpu


def operands(N, K, f16, seed):
    r = np.random.default_rng(seed)
    A, B = r.standard_normal(K).astype(np.float32), (0.02 * r.standard_normal((K, N))).astype(np.float32)
    B = B.astype(np.float16).astype(np.float32) if f16 else B
    return A, B, r.standard_normal(N).astype(np.float32), r.standard_normal(N).astype(np.float32)


def exact(A, B, bias, res):
    return A.astype(np.float64) @ B.astype(np.float64) + bias + res


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("N,K", [(1, 1), (3, 300), (7, 257), (9, 1023), (33, 64), (17, 2049), (515, 6400), (1601, 3000),
                                 (2563, 100), (10243, 65), (20487, 33)])
def test_matvec_edges(g2, N, K, f16):
    A, B, bias, res = operands(N, K, f16, N + K)
    dA, dbias = g2.to_device(A), g2.to_device(bias)
    raw = g2.convert_f16(B) if f16 else B
    bound = dot_bound(np.abs(A), np.abs(B), K)
    for shift in (0, raw.itemsize):  # B at a vector's address, then one element past it
        dB = g2.to_device(np.concatenate([np.zeros(shift // raw.itemsize, raw.dtype), raw.ravel()]))
        dC = g2.to_device(np.concatenate([res, np.full(8, 7.0, np.float32)]))
        g2.matvec(dA, dB.offset(shift), dbias, dC, dC, N, K, f16=f16)
        got = dC.download(np.float32, N + 8)
        assert (got[N:] == 7.0).all()  # nothing past the vector
        assert_close_bound(got[:N], exact(A, B, bias, res), bound, what="matvec")


LARGE = [(False, 6301, 2050), (False, 9001, 2049), (False, 3126, 4100), (True, 10007, 2600), (True, 12505, 2049)]


@pytest.mark.parametrize("f16,N,K", LARGE)
def test_matvec_large(g2, f16, N, K):
    """Matrices of 50 MB and more with long columns: 64, 16 and 8 lanes to a
    work-group, in K slices that do not divide K, ragged columns; GELU and
    residual behind the slices."""
    A, B, bias, res = operands(N, K, f16, N)
    dC = g2.to_device(np.concatenate([res, np.full(8, 7.0, np.float32)]))
    g2.matvec(g2.to_device(A), g2.to_device(g2.convert_f16(B) if f16 else B), g2.to_device(bias), dC, dC, N, K, f16=f16)
    got = dC.download(np.float32, N + 8)
    assert (got[N:] == 7.0).all()
    assert_close_bound(got[:N], exact(A, B, bias, res), dot_bound(np.abs(A), np.abs(B), K), what="matvec")


@pytest.mark.parametrize("N,K", [(768, 768), (100, 2500)])
def test_matvec_in_place(g2, N, K):
    """C in A's memory: the product reads all of A first."""
    A, B, bias, res = operands(N, K, False, 9)
    dA = g2.to_device(A)
    g2.matvec(dA, g2.to_device(B), g2.to_device(bias), g2.to_device(res), dA, N, K)
    assert_close_bound(dA.download(np.float32, N), exact(A, B, bias, res), dot_bound(np.abs(A), np.abs(B), K), what="in place")


@pytest.mark.parametrize("N", [33, 64])
@pytest.mark.parametrize("shift", [-1, 1, 16])
def test_matvec_over_a_shifted_residual(g2, N, shift):
    """Up to 64 columns, a wave's, over the residual or the bias a few elements on."""
    A, B, bias, res = operands(N, 300, False, 8)
    ref, bound = exact(A, B, bias, res), dot_bound(np.abs(A), np.abs(B), 300)
    pad = np.zeros(16, np.float32)
    for which in (0, 1):
        held = g2.to_device(np.concatenate([pad, (bias, res)[which], pad]))
        other = g2.to_device((res, bias)[which])
        pair = (held.offset(64), other) if which == 0 else (other, held.offset(64))
        g2.matvec(g2.to_device(A), g2.to_device(B), *pair, held.offset(64 + 4 * shift), N, 300)
        got = held.download(np.float32, N + 32)[16 + shift:][:N]
        assert_close_bound(got, ref, bound, what="shifted")


@pytest.mark.parametrize("N,K", [(256, 256), (64, 700), (128, 128)])
def test_matvec_sk_in_place(g2, N, K):
    """One slice over A, up to 256 columns."""
    A, B, _, _ = operands(N, K, False, 10)
    dA = g2.to_device(A)
    g2.matvec_sk(dA, g2.to_device(B), dA, N, K, 1)
    assert_close_bound(dA.download(np.float32, N), exact(A, B, 0, 0), dot_bound(np.abs(A), np.abs(B), K), what="in place")


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("N,K,ks", [(4, 3, 8), (12, 2, 5), (36, 1025, 3), (1028, 700, 7), (2564, 6400, 8)])
def test_matvec_sk_edges(g2, N, K, ks, f16):
    A, B, _, _ = operands(N, K, f16, N + K + ks)
    dP = g2.to_device(np.full(ks * N + 8, 7.0, np.float32))
    g2.matvec_sk(g2.to_device(A), g2.to_device(g2.convert_f16(B) if f16 else B), dP, N, K, ks, f16=f16)
    got = dP.download(np.float32, ks * N + 8)
    assert (got[ks * N:] == 7.0).all()
    ref = oracle.matvec4_sk(A, B, N, K, ks)
    for s in range(ks):
        bound = dot_bound(np.abs(A[s::ks]), np.abs(B[s::ks]), max(len(A[s::ks]), 1))
        assert_close_bound(got[s * N:(s + 1) * N], ref[s], bound, what=f"slice {s}")


@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
def test_matvec_sk_wider_than_a_launch(g2, f16):
    """2^28 + 4 columns (16 threads each would be 2^32): several launches,
    whose last has fewer columns than an fp16 vector."""
    N = (1 << 28) + 4
    B = np.arange(N, dtype=np.uint32).astype(np.uint16) % 1000
    B = (g2.convert_f16(np.arange(1000, dtype=np.float32)) if f16 else np.arange(1000, dtype=np.float32))[B]
    dP = g2.DevBuf(4 * N)
    g2.matvec_sk(g2.to_device(np.float32([3.0])), g2.to_device(B), dP, N, 1, 1, f16=f16)
    got = dP.download(np.float32, N)
    want = B.view(np.float16).astype(np.float32) if f16 else B
    assert (got == 3 * want).all()


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1025, 4097])
def test_elementwise_tails(g2, n):
    """add and gelu, four elements to a thread: every remainder, one element
    past an aligned address, nothing past the end."""
    r = np.random.default_rng(n)
    a, b = (r.standard_normal(n + 2).astype(np.float32) for _ in range(2))
    da, db = g2.to_device(a), g2.to_device(b)
    g2.add(da.offset(4), db.offset(4), n)
    np.testing.assert_array_equal(da.download(np.float32, n + 2), np.concatenate([a[:1], a[1:-1] + b[1:-1], a[-1:]]))
    g2.gelu(db.offset(4), n)
    got = db.download(np.float32, n + 2)
    np.testing.assert_allclose(got[1:-1], oracle.gelu(b[1:-1].copy()), rtol=4e-6, atol=1e-6)
    assert got[0] == b[0] and got[-1] == b[-1]


@pytest.mark.parametrize("E", [1, 255, 257, 2047, 2048, 2049, 5000])
def test_layernorm_widths(g2, E):
    """Rows kept in registers (up to 2048) and rows read three times."""
    r = np.random.default_rng(E)
    x, g, b = r.standard_normal((3, E)).astype(np.float32) * 3 + 0.5, *r.standard_normal((2, E)).astype(np.float32)
    dO = g2.to_device(np.full(3 * E + 4, 7.0, np.float32))
    g2.layernorm(g2.to_device(x), dO, g2.to_device(g), g2.to_device(b), E, 3)
    got = dO.download(np.float32, 3 * E + 4)
    np.testing.assert_allclose(got[:3 * E].reshape(3, E), oracle.layernorm(x, g, b, E, 3), rtol=2e-5, atol=2e-5)
    assert (got[3 * E:] == 7.0).all()
