"""The small tiles of fp32 products on split operands (kernels/gemm_mfma_split.hip.h: config_small) beyond the whole 64 x 64 ones: guarded
ones and those of 64 x 96 and 96 x 64, in every layout through the library call, and through programs.  Bounds as in test_split_gemm.py."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from test_split_gemm import PROGRAMS, allowed_distance, bound, call, distance, operands
from tiramisu_amd import build, runtime


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('''#include "%s"
extern "C" int tile(long M, long N, long K, int aligned, int split_rows) {
    const ttarget::fp32_tiles t = ttarget::library_tiles_for(M, N, K, 1, aligned);
    const ttarget::split_tile s = ttarget::any_split_tile_for(M, N, K, 1, t.m, t.n, t.guarded, split_rows);
    return 1000 * s.m + s.n;
}
extern "C" int square(long M, long N, long K, int aligned) {
    const ttarget::fp32_tiles t = ttarget::library_tiles_for(M, N, K, 1, aligned);
    return ttarget::split_tile_for(M, N, K, 1, t.m, t.n, t.guarded);
}
extern "C" int lds(int m, int n, int a, int b) { return ttarget::split_lds_bytes(m, n, a, b); }
''' % os.path.join(build.CSRC, "kernels", "target_gfx950.h"))
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "rule.so"), str(d / "rule.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "rule.so"))
    lib.square.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int]
    lib.tile.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int] * 2
    return lib


def test_rule(rule):
    assert rule.tile(4096, 4096, 4096, True, False) == 256256 and rule.tile(1024, 1024, 1024, True, False) == 64064 and rule.tile(512, 512, 512, True, False) == 0
    assert rule.tile(737, 894, 2361, True, False) == 64064 and rule.tile(737, 894, 2361, True, True) == 0
    rng = np.random.RandomState(1)
    for _ in range(3000):
        M, N, K = (int(v) for v in np.exp(rng.uniform(np.log(16), np.log(5000), 3)))
        aligned = rng.rand() < 0.7
        tile, square = rule.tile(M, N, K, aligned, K % 4 != 0), rule.square(M, N, K, aligned)
        if tile == 0:
            assert square == 0                             # no product leaves the split operands
        else:      # sizes that the kernels' loads require
            assert min(M, N) >= 64 and K >= 96 and (tile in (64064, 64096, 96064) or tile == 1001 * square)
    for a in (0, 1):
        for b in (0, 1):
            assert all(rule.lds(m, n, a, b) <= 160 * 1024 for m, n in ((64, 64), (64, 96), (96, 64), (128, 128), (256, 256)))


SIZES = [(446, 1497, 733, 64064), (1705, 445, 642, 64064), (1001, 1503, 703, 64096), (353, 3041, 419, 64096), (1503, 1001, 703, 96064), (1024, 1344, 176, 64096),
         (1344, 1024, 176, 96064), (1024, 1536, 704, 64096)]


@pytest.mark.gpu
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,tile", SIZES)
def test_library_call(rule, M, N, K, tile, tA, tB):
    assert rule.tile(M, N, K, True, False) == tile
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
            assert distance(out[:, :N], expected) <= allowed_distance(K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(446, 1497, 733), (1001, 1503, 703), (1344, 1024, 176)])
@pytest.mark.parametrize("transposed", [False, True])
def test_numbers_that_three_parts_do_not_hold(M, N, K, transposed):
    """A wavefront that finds sums that are not finite computes its k again with the fp32 instruction: in the first and last rows,
    columns and k, beyond the scale and below it.  (Bounds of test_split_gemm.py's test of that name.)"""
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
@pytest.mark.parametrize("M,N,K,tile", [(446, 1497, 733, "64x64x64, guarded"), (1001, 1503, 703, "64x96x64, guarded"), (1344, 1024, 176, "96x64x64, whole")])
def test_program(M, N, K, tile):
    p = runtime.load(PROGRAMS, "sgemm_%dx%dx%d" % (M, N, K))
    assert any("three bf16 parts" in k["how"] and "tile " + tile in k["how"] for k in p.manifest["kernels"])
    from gpu_util import DeviceArray
    rng = np.random.RandomState(K)
    A, B, C = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32), rng.uniform(-1, 1, (M, N)).astype(np.float32)
    d = [DeviceArray(x) for x in (A, B, C)]
    p(np.array([1.5, 0.5], np.float32), *[x.buffer() for x in d])
    a, b = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(d[2].download() - (1.5 * (a @ b) + 0.5 * C)) <= 1.5 * bound(a, b, K) + 2.0 ** -23)
