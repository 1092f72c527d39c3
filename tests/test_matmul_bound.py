"""The accuracy bound of test_matmul_gpu.py, on the CPU: the six products of
bf16 parts that the GEMM sums stay well inside it, and it is broken when the
third parts' products, or the second parts' product, are missing."""
import numpy as np
import pytest

from test_matmul_gpu import sum_bound


def bf16(v):
    u = v.astype(np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


def parts(v):
    out = []
    for _ in range(3):
        p = bf16(v)
        out.append(p.astype(np.float64))
        v = (v - p).astype(np.float32)
    assert not v.any()  # three parts are all of an fp32 value
    return out


@pytest.mark.parametrize("K", [70, 300, 1389, 4100])
def test_bound_notices_a_missing_part(K):
    r = np.random.default_rng(K)
    A, B = r.standard_normal((24, K)).astype(np.float32), r.standard_normal((K, 200)).astype(np.float32)
    a, b = parts(A), parts(B)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    six = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]

    def error(pairs):
        return np.linalg.norm(sum(a[i] @ b[j] for i, j in pairs) - ref) / np.linalg.norm(ref)

    assert error(six) < sum_bound(K) / 4
    for missing in ((0, 2), (2, 0), (1, 1)):
        assert error([p for p in six if p != missing]) > sum_bound(K), missing
