"""fp32 products of some hundred rows and columns that no square of split operands (kernels/gemm_mfma_split.hip.h) covers well: with the fp32
instruction, in every layout through the library call, and through programs.

Small whole numbers are exact.  With uniform operands the accumulator is rounded once per matrix instruction, of two k, each time by at most
2^-24 of the sum of the magnitudes so far, half the final one on average: |error| <= (K / 2 / 2 2^-24) sum |a b|, with a few more roundings for
partial sums, alpha and beta."""
import numpy as np
import pytest

from test_split_gemm import PROGRAMS, call, operands, rule  # noqa: F401
from tiramisu_amd import runtime


def bound(A, B, K):
    return (K / 4 + 24) * 2.0 ** -24 * (np.abs(A) @ np.abs(B))


SIZES = [(446, 1497, 733), (1705, 445, 642), (1001, 1503, 703), (353, 3041, 419), (1503, 1001, 703), (1024, 1344, 176), (1344, 1024, 176), (1024, 1536, 704)]


@pytest.mark.gpu
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_library_call(rule, M, N, K, tA, tB):
    assert rule.split_tile(M, N, K, True) == 0
    rng = np.random.RandomState(M + K)
    for kind, pad, offset, alpha, beta in (("whole", 0, 0, 2.0, 3.0), ("uniform", 3, 1, 1.0, 0.0)):
        A, B = operands(rng, M, N, K, tA, tB, pad, kind)
        a, b = (A[:, :M].T if tA else A[:, :K]).astype(np.float64), (B[:, :K].T if tB else B[:, :N]).astype(np.float64)
        C = rng.randint(-8, 9, (M, N + pad)).astype(np.float32)
        out = call(A, B, C, M, N, K, alpha, beta, tA, tB, offset)
        expected = alpha * (a @ b) + beta * C[:, :N]
        assert np.array_equal(out[:, N:], C[:, N:])
        if kind == "whole":
            assert np.array_equal(out[:, :N], expected)
        else:
            assert np.all(np.abs(out[:, :N] - expected) <= bound(a, b, K))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(446, 1497, 733), (1001, 1503, 703), (1344, 1024, 176)])
@pytest.mark.parametrize("transposed", [False, True])
def test_numbers_that_three_parts_do_not_hold(M, N, K, transposed):
    """Infinities, NaN and numbers beyond the scale of split operands and below it: in the first and last rows, columns and k."""
    rng = np.random.RandomState(5)
    A, B = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    A[3, 5], A[M - 1, K - 1], A[70, 0], B[7, 9], B[K - 1, N - 1] = np.inf, np.nan, 2.0 ** 120, -np.inf, np.inf
    A[130] *= np.float32(2.0 ** 115)
    B[:, 200] *= np.float32(2.0 ** -100)
    A[132] *= np.float32(2.0 ** -126)
    with np.errstate(all="ignore"):
        expected = A.astype(np.float64) @ B.astype(np.float64)
        fp32 = expected.astype(np.float32)
        a, b = (np.ascontiguousarray(x.T) for x in (A, B)) if transposed else (A, B)
        out = call(a, b, np.zeros((M, N), np.float32), M, N, K, 1.0, 0.0, transposed, transposed)
        assert np.array_equal(np.isnan(out), np.isnan(fp32)) and np.array_equal(np.isinf(out), np.isinf(fp32))
        assert np.array_equal(np.sign(out[np.isinf(out)]), np.sign(fp32[np.isinf(out)]))
        fine = np.isfinite(fp32)
        finite = lambda x: np.where(np.isfinite(x), x, 0).astype(np.float64)
        allowed = (K + 24) * 2.0 ** -24 * (np.abs(finite(A)) @ np.abs(finite(B))) + 2.0 ** -149 * K
        assert np.all(np.abs(out[fine] - expected[fine]) <= allowed[fine])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(446, 1497, 733), (1001, 1503, 703), (1344, 1024, 176)])
def test_program(M, N, K):
    p = runtime.load(PROGRAMS, "sgemm_%dx%dx%d" % (M, N, K))
    assert any("v_mfma_f32_32x32x2_f32" in k["how"] for k in p.manifest["kernels"])
    from gpu_util import DeviceArray
    rng = np.random.RandomState(K)
    A, B, C = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32), rng.uniform(-1, 1, (M, N)).astype(np.float32)
    d = [DeviceArray(x) for x in (A, B, C)]
    p(np.array([1.5, 0.5], np.float32), *[x.buffer() for x in d])
    a, b = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(d[2].download() - (1.5 * (a @ b) + 0.5 * C)) <= 1.5 * bound(a, b, K) + 2.0 ** -23)
