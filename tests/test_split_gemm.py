"""fp32 products whose operands are split into bf16 parts (kernels/gemm_mfma_split.hip.h): the rule that picks them on the CPU,
and on the GPU every tile, whole and guarded, in every layout, through the library call and the programs.

Exactness: products and sums of small whole numbers are exact.  Accuracy: with uniform operands a sum of K products rounds its
accumulator once per matrix instruction, six per sixteen k, each time by at most 2^-24 of the sum of the magnitudes so far; the
products left out are below 2^-24 of theirs.  |error| <= (6/16 K 2^-24 / 2 + 2^-24) sum |a b| therefore bounds every element (on
average half the accumulator's final value is there when it is rounded), with a few more roundings for partial sums, alpha and beta.
One product per sum: see test_one_product_per_sum.

The whole result, by the 2-norm: each rounding is off by 2^-23 / sqrt(12) of the accumulator's size on average, and that size grows with
the root of k: 6/16 K roundings come to sqrt(3/16 K / 12) 2^-23 = sqrt(K) / 8 2^-23 of the result.  Twice that, and 2^-24 for the products left
out, is allowed: at most 8e-7 at the sizes here, where any one of the six products missing is off by 2e-6 (see test_missing_products)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tiramisu_amd import build, runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAMS = os.path.join(ROOT, "tests", "programs")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """split_tile_for of kernels/target_gfx950.h, preceded by the fp32 tile that the library call would take."""
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('''#include "%s"
extern "C" int fp32_tile(long M, long N, long K, int aligned, int *m, int *n) {
    const ttarget::fp32_tiles t = ttarget::library_tiles_for(M, N, K, 1, aligned);
    *m = t.m;
    *n = t.n;
    return t.guarded;
}
extern "C" int split_tile(long M, long N, long K, int aligned) {
    const ttarget::fp32_tiles t = ttarget::library_tiles_for(M, N, K, 1, aligned);
    return ttarget::split_tile_for(M, N, K, 1, t.m, t.n, t.guarded);
}
extern "C" double fp32_model(long M, long N, long K, int m, int n, int guarded) {
    for (const ttarget::launch_model &l : ttarget::FP32_LAUNCHES)
        if (l.m == m && l.n == n && l.guarded == (bool)guarded) return ttarget::modelled(l, M, N, K, 1);
    return 0;
}
''' % os.path.join(build.CSRC, "kernels", "target_gfx950.h"))
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "rule.so"), str(d / "rule.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "rule.so"))
    sizes, out = [ctypes.c_long] * 3, [ctypes.POINTER(ctypes.c_int)] * 2
    lib.split_tile.argtypes, lib.fp32_tile.argtypes = sizes + [ctypes.c_int], sizes + [ctypes.c_int] + out
    lib.fp32_model.argtypes, lib.fp32_model.restype = sizes + [ctypes.c_int] * 3, ctypes.c_double
    return lib


def test_rule(rule):
    for M, N, K, edge in ((4096, 4096, 4096, 256), (2048, 2048, 2048, 128), (1024, 1024, 1024, 64), (4096, 4096, 95, 0), (63, 4096, 4096, 0),
                          (4096, 63, 4096, 0), (512, 512, 512, 0), (64, 64, 4096, 0), (4097, 4096, 96, 256),
                          # a square tile of 256 or 192 that K asks to guard: the library's fp32 tiles are 64 x 64
                          (4096, 4096, 1000, 256), (4096, 4096, 4095, 256), (3072, 3072, 3000, 128), (3840, 3840, 500, 256)):
        assert rule.split_tile(M, N, K, True) == edge, (M, N, K)
    assert rule.split_tile(4096, 4096, 4096, False) == 256
    m, n = ctypes.c_int(), ctypes.c_int()
    rng = np.random.RandomState(1)
    for _ in range(3000):
        M, N, K = (int(v) for v in np.exp(rng.uniform(np.log(16), np.log(5000), 3)))
        if rng.rand() < 0.5:
            M, N, K = (max(64, v // 64 * 64) for v in (M, N, K))
        aligned = rng.rand() < 0.7
        edge = rule.split_tile(M, N, K, aligned)
        guarded = rule.fp32_tile(M, N, K, aligned, m, n)
        assert rule.fp32_model(M, N, K, m, n, guarded) > 0            # every tile that the library launches has its figures
        if edge:      # sizes that the kernels' loads require; as many partial sums as the fp32 tile's four, or more
            assert min(M, N) >= 64 and K >= 96 and (n.value != 32 or edge == 64)
            assert edge != 64 or (M % 64 == 0 and N % 64 == 0 and K % 16 == 0)


def bound(A, B, K):
    return (6 / 16 * K / 2 + 24) * 2.0 ** -24 * (np.abs(A) @ np.abs(B)) + 2.0 ** -24 * (np.abs(A) @ np.abs(B))


def distance(out, expected):
    return np.linalg.norm(out - expected) / np.linalg.norm(expected)


def allowed_distance(K):
    return 2 * K ** 0.5 / 8 * 2.0 ** -23 + 2.0 ** -24


def test_missing_products():
    """Five of the six products, in 64 bits: every one that is left out shows in the distance that the tests allow."""
    def bf16(x):
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)

    def parts(x):
        h = bf16(x)
        m = bf16(x - h)
        return [p.astype(np.float64) for p in (h, m, x - h - m)]

    rng = np.random.RandomState(6)
    K = max([s[2] for s in SIZES] + [32 * 9])
    A, B = (parts(rng.uniform(-1, 1, s).astype(np.float32)) for s in ((64, K), (K, 64)))
    six = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]
    expected = sum(A) @ sum(B)
    assert distance(sum(A[i] @ B[j] for i, j in six), expected) < 2.0 ** -24
    for left_out in six:
        assert distance(sum(A[i] @ B[j] for i, j in six if (i, j) != left_out), expected) > 1.5 * allowed_distance(K)


def operands(rng, M, N, K, tA, tB, pad, kind):
    def one(rows, cols):
        full = np.full((rows, cols + pad), np.nan, np.float32)       # what lies between the rows must not matter
        full[:, :cols] = rng.randint(-8, 9, (rows, cols)) if kind == "whole" else rng.uniform(-1, 1, (rows, cols))
        return full
    return one(*((K, M) if tA else (M, K))), one(*((N, K) if tB else (K, N)))


def call(A, B, C, M, N, K, alpha, beta, tA, tB, offset=0):
    from gpu_util import DeviceArray
    dA, dB, dC = (DeviceArray(np.concatenate([np.zeros(offset, np.float32), x.ravel()])) for x in (A, B, C))
    rc = runtime.wrappers().tiramisu_hip_sgemm(dA.ptr, dB.ptr, dC.ptr, M, N, K, alpha, beta, A.shape[1], B.shape[1], C.shape[1], offset, offset, offset, tA, tB)
    assert rc == 0
    return dC.download()[offset:].reshape(C.shape)


def test_lanes_that_share_lds_without_a_barrier_are_ordered(tmp_path):
    """64 x 64 tiles pass a slice from lane to lane through LDS without a barrier of the workgroup.  Seen per thread the addresses stored to
    and read from differ, so only a fence keeps the compiler from moving one across the other: in what it makes of the kernel, every
    run of stores to LDS stands between two fences."""
    source, ir = tmp_path / "waves.hip", tmp_path / "waves.ll"
    source.write_text('#include "gemm_mfma_split.hip.h"\n' + "".join(
        "template __global__ void tgemm::sgemm_split_kernel<tgemm::config_waves<%s, %s>>(const float *, const float *, float *, int, int, int, long, long, long,"
        " float, float);\n" % layout for layout in (("true", "false"), ("false", "true"))))
    subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["-w", "--cuda-device-only", "-S", "-emit-llvm", "-I" + os.path.join(build.CSRC, "kernels"), str(source), "-o", str(ir)], check=True)
    runs, before = 0, None                # the last fence ("fence") or access to LDS ("load", "store") of the block
    for line in ir.read_text().splitlines():
        text = line.strip()
        if line[:1] not in (" ", "\t") and before is not None:
            assert before != "store", "a block ends behind stores"
            before = None
        elif text.startswith("fence "):
            before = "fence"
        elif "addrspace(3)" in text and text.startswith("store "):
            assert before in ("fence", "store"), text
            runs += before == "fence"
            before = "store"
        elif "addrspace(3)" in text and " = load " in text:
            assert before != "store", text
            before = "load"
    assert runs >= 2 * 3                  # the first slice, two stages of the loop, in two kernels


SIZES = [(704, 1088, 528, 64), (1408, 2560, 416, 128), (1219, 2747, 611, 128), (1300, 2690, 450, 128), (2560, 3584, 208, 256), (2701, 3915, 99, 256),
         (2560, 3584, 210, 256)]        # (all but K a multiple of the tile)


@pytest.mark.gpu
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,edge", SIZES)
def test_library_call(rule, M, N, K, edge, tA, tB):
    assert rule.split_tile(M, N, K, True) == rule.split_tile(M, N, K, False) == edge
    rng = np.random.RandomState(M + K)
    for kind, pad, offset, alpha, beta in (("whole", 0, 0, 2.0, 3.0), ("uniform", 3 if edge != 64 else 4, 1 if M % 2 else 4, 1.0, 0.0)):
        A, B = operands(rng, M, N, K, tA, tB, pad, kind)
        a = A[:, :M].T if tA else A[:, :K]
        b = B[:, :K].T if tB else B[:, :N]
        C = rng.randint(-8, 9, (M, N + pad)).astype(np.float32)
        out = call(A, B, C, M, N, K, alpha, beta, tA, tB, offset)
        a, b = a.astype(np.float64), b.astype(np.float64)
        expected = alpha * (a @ b) + beta * C[:, :N]
        assert np.array_equal(out[:, N:], C[:, N:])
        if kind == "whole":
            assert np.array_equal(out[:, :N], expected)
        else:
            assert np.all(np.abs(out[:, :N] - expected) <= bound(a, b, K))
            assert distance(out[:, :N], expected) <= allowed_distance(K)


# Sums of one product each: the parts of both operands show one by one.
#   random   the five smaller products add up to at most 2^-7 of the product before the largest joins them: their roundings are
#            below 5 2^-31 of it, 2^-5 units in the last place.  Then one rounding, half a unit, and what is left out, below
#            2^-24 of the product: less than a unit.
#   others   the product has 24 significant bits at most, of 24 times one (all three parts of one operand) or of 12 times
#            12 (hA*hB, hA*mB, mA*hB, mA*mB): exact, and every partial sum with it.
LONE = ("random", "long times one", "one times long", "half times half")


def lone_operands(rng, kind, a_shape, b_shape):
    """Positive numbers for the two operands."""
    draw = {"random": lambda s: rng.uniform(0.5, 2, s), "long": lambda s: rng.randint(1 << 22, 1 << 23, s) * 2 + 1,
            "one": lambda s: 2.0 ** rng.randint(-20, 20, s), "half": lambda s: rng.randint(1 << 10, 1 << 11, s) * 2 + 1}
    names = ("random", "random") if kind == "random" else kind.split(" times ")
    return [draw[n](s).astype(np.float32) for n, s in zip(names, (a_shape, b_shape))]


def check_lone(out, expected, kind):
    if kind == "random":
        assert np.all(np.abs(out - expected) <= (1.5 + 2.0 ** -5) * np.spacing(expected.astype(np.float32)))
    else:
        assert np.array_equal(out, expected)


@pytest.mark.gpu
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,edge", SIZES)
def test_one_product_per_sum(rule, M, N, K, edge, tA, tB):
    assert rule.split_tile(M, N, K, True) == rule.split_tile(M, N, K, False) == edge
    rng = np.random.RandomState(K)
    for kind in LONE:
        at = rng.permutation(M) % K                       # (M > K: every k has its rows)
        values, b = lone_operands(rng, kind, M, (K, N))
        a = np.zeros((M, K), np.float32)
        a[np.arange(M), at] = values
        out = call(np.ascontiguousarray(a.T) if tA else a, np.ascontiguousarray(b.T) if tB else b, np.zeros((M, N), np.float32), M, N, K, 1.0, 0.0, tA, tB)
        check_lone(out, values[:, None].astype(np.float64) * b[at], kind)


@pytest.mark.gpu
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(1000, 1500, 700), (446, 1497, 733), (1001, 1503, 703), (1344, 1024, 176)])
def test_products_of_the_fp32_instruction_are_rounded_once(rule, M, N, K, tA, tB):
    """Sizes whose fp32 tiles are 64 x 32 or 32 x 32: no square of the split operands has as many partial sums there, and six of nine partial
    products would not do instead: one product alone, exact in 64 bits, comes out rounded to fp32 once, to nearest."""
    assert rule.split_tile(M, N, K, True) == 0
    rng = np.random.RandomState(K)
    at = rng.permutation(M) % K
    values, b = lone_operands(rng, "random", M, (K, N))
    a = np.zeros((M, K), np.float32)
    a[np.arange(M), at] = values
    out = call(np.ascontiguousarray(a.T) if tA else a, np.ascontiguousarray(b.T) if tB else b, np.zeros((M, N), np.float32), M, N, K, 1.0, 0.0, tA, tB)
    assert np.array_equal(out, (values[:, None].astype(np.float64) * b[at]).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [s[:3] for s in SIZES if s[0] != 1300])
def test_program(M, N, K):
    name = "sgemm_%dx%dx%d" % (M, N, K)
    p = runtime.load(PROGRAMS, name)
    assert any("three bf16 parts" in k["how"] for k in p.manifest["kernels"])
    from gpu_util import DeviceArray
    rng = np.random.RandomState(K)
    A, B, C = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32), rng.uniform(-1, 1, (M, N)).astype(np.float32)
    d = [DeviceArray(x) for x in (A, B, C)]
    p(np.array([1.5, 0.5], np.float32), *[x.buffer() for x in d])
    a, b = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(d[2].download() - (1.5 * (a @ b) + 0.5 * C)) <= 1.5 * bound(a, b, K) + 2.0 ** -23)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(704, 1088, 528), (1219, 2747, 611), (2560, 3584, 208), (2701, 3915, 99)])
@pytest.mark.parametrize("transposed", [False, True])         # (each operand in both layouts)
def test_numbers_that_three_parts_do_not_hold(M, N, K, transposed):
    rng = np.random.RandomState(5)
    A, B = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    A[3, 5], A[M - 1, K - 1], A[70, 0], B[7, 9] = np.inf, np.nan, 2.0 ** 120, -np.inf
    A[130] *= np.float32(2.0 ** 115)                        # a row of large numbers: beyond the scale, their sums well within range
    B[:, 200] *= np.float32(2.0 ** -100)
    A[131] = np.float32(2.0 ** -120) * A[131]               # products down to 2^-240: zero or subnormal
    A[132] *= np.float32(2.0 ** -126)                       # subnormal numbers, against columns of ordinary ones
    with np.errstate(all="ignore"):
        expected = A.astype(np.float64) @ B.astype(np.float64)
        fp32 = expected.astype(np.float32)
        a, b = (np.ascontiguousarray(x.T) for x in (A, B)) if transposed else (A, B)
        out = call(a, b, np.zeros((M, N), np.float32), M, N, K, 1.0, 0.0, transposed, transposed)
        assert np.array_equal(np.isnan(out), np.isnan(fp32))
        # (a sum of fp32 numbers may overflow where the exact one does not: only near the largest number, which no element is)
        assert np.array_equal(np.isinf(out), np.isinf(fp32)) and np.array_equal(np.sign(out[np.isinf(out)]), np.sign(fp32[np.isinf(out)]))
        fine = np.isfinite(fp32)
        finite = lambda x: np.where(np.isfinite(x), x, 0).astype(np.float64)
        # (the fp32 instruction's bound where a tile was computed again: 16 roundings per 16 k)
        allowed = (K + 24) * 2.0 ** -24 * (np.abs(finite(A)) @ np.abs(finite(B))) + 2.0 ** -149 * K
        assert np.all(np.abs(out - expected)[fine] <= allowed[fine])


@pytest.mark.gpu
def test_batch_scope_is_one_launch_of_split_tiles():
    from gpu_util import DeviceArray
    M, N, K, n = 640, 640, 640, 5
    rng = np.random.RandomState(2)
    A, B = rng.randint(-8, 9, (n, M, K)).astype(np.float32), rng.randint(-8, 9, (n, K, N)).astype(np.float32)
    dA, dB, dC = DeviceArray(A), DeviceArray(B), DeviceArray(np.zeros((n, M, N), np.float32))
    w = runtime.wrappers()
    assert w.tiramisu_hip_batch_begin() == 0
    for i in range(n):
        w.tiramisu_hip_sgemm(dA.ptr + 4 * i * M * K, dB.ptr + 4 * i * K * N, dC.ptr + 4 * i * M * N, M, N, K, 1.0, 0.0, 0, 0, 0, 0, 0, 0, False, False)
    assert w.tiramisu_hip_batch_end() == 0
    assert np.array_equal(dC.download(), A.astype(np.float64) @ B.astype(np.float64))


def conv_expected(x, w, bias):
    """Convolution plus bias and the sum of the magnitudes, in float64, image by image (x padded)."""
    n, ci, hp, wp = x.shape
    co, h = w.shape[0], hp - 2
    out, size = (np.empty((n, co, h, h)) for _ in range(2))
    w2 = w.reshape(co, -1).astype(np.float64)
    for i in range(n):
        cols = np.stack([x[i, :, ky:ky + h, kx:kx + h] for ky in range(3) for kx in range(3)], 1).reshape(ci * 9, h * h).astype(np.float64)
        with np.errstate(all="ignore"):
            out[i] = (w2 @ cols).reshape(co, h, h) + bias[:, None, None]
            size[i] = (np.abs(w2) @ np.abs(cols)).reshape(co, h, h) + np.abs(bias)[:, None, None]
    return out, size


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["whole", "uniform", "special"])
def test_windowed_convolution(kind):
    from gpu_util import DeviceArray
    name, shape = "conv2d_9x32x64x128", (9, 32, 64, 128)
    p = runtime.load(PROGRAMS, name)
    how = [k["how"] for k in p.manifest["kernels"]]
    assert any("three bf16 parts" in s and "sliding window" in s and "cut into" in s for s in how)
    n, ci, co, h = shape
    rng = np.random.RandomState(3)
    x, w, bias = np.zeros((n, ci, h + 2, h + 2), np.float32), rng.uniform(-1, 1, (co, ci, 3, 3)).astype(np.float32), rng.uniform(-1, 1, co).astype(np.float32)
    x[:, :, 1:-1, 1:-1] = rng.uniform(-1, 1, (n, ci, h, h))
    if kind == "whole":
        x, w, bias = (np.round(8 * v).astype(np.float32) for v in (x, w, bias))
    if kind == "special":        # in a whole tile, in a piece, and small numbers
        x[0, 5, 40, 40], x[8, 31, 128, 100], x[4] = np.inf, np.nan, x[4] * np.float32(2.0 ** -126)
    d = [DeviceArray(v) for v in (x, w, bias, np.zeros((n, co, h, h), np.float32))]
    p(*[v.buffer() for v in d])
    out = d[3].download()
    expected, size = conv_expected(x, w, bias)
    relu = np.where(np.isnan(expected), 0.0, np.maximum(expected, 0))
    if kind == "whole":
        assert np.array_equal(out, relu)
        return
    fine = np.isfinite(expected)
    K = ci * 9
    allowed = (K + 24) * 2.0 ** -24 * size + 2.0 ** -149 * K if kind == "special" else (6 / 16 * K / 2 + 24) * 2.0 ** -24 * size + 2.0 ** -24 * size
    assert np.all(np.abs(out - relu)[fine] <= allowed[fine])
    if kind == "uniform":
        positive = expected > 0                           # (the others are zero)
        assert distance(out[positive], expected[positive]) <= allowed_distance(K)
    assert np.array_equal(np.isinf(out), expected == np.inf)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", LONE)
def test_windowed_convolution_of_one_product_per_sum(kind):
    from gpu_util import DeviceArray
    n, ci, co, h = 9, 32, 64, 128
    p = runtime.load(PROGRAMS, "conv2d_9x32x64x128")
    rng = np.random.RandomState(4)
    x = np.zeros((n, ci, h + 2, h + 2), np.float32)
    values, x[:, :, 1:-1, 1:-1] = lone_operands(rng, kind, ci * 9, (n, ci, h, h))
    dx, dbias, dout = DeviceArray(x), DeviceArray(np.zeros(co, np.float32)), DeviceArray(np.zeros((n, co, h, h), np.float32))
    places = np.concatenate([rng.permutation(ci * 9), rng.permutation(ci * 9)])
    for first in range(0, ci * 9, co):                    # every input channel and tap has an output channel
        at = places[first:first + co]
        w = np.zeros((co, ci * 9), np.float32)
        w[np.arange(co), at] = values[at]
        dw = DeviceArray(w.reshape(co, ci, 3, 3))
        p(dx.buffer(), dw.buffer(), dbias.buffer(), dout.buffer())
        out = dout.download()
        for o in range(co):
            c, ky, kx = at[o] // 9, at[o] % 9 // 3, at[o] % 3
            check_lone(out[:, o], x[:, c, ky:ky + h, kx:kx + h].astype(np.float64) * values[at[o]], kind)
