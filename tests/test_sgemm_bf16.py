"""bf16-input / fp32-accumulate sgemm (the bf16 variant of benchmark configuration 3).

The reference has no bf16 type, so the oracle is the fp32 result on bf16-rounded inputs
(round to nearest even), as computed by the CPU-generated code of the same program and by
float64 numpy.  Products of two bf16 numbers are exact in fp32, so only the summation order
differs between paths: tolerance max |gpu - ref| <= 2e-2 * max |ref| (the parity statement's
bf16 bound); integer-valued data is exact."""
import os

import numpy as np
import pytest

from oracle import build as oracle_build
from tiramisu_amd import runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAMS = os.path.join(ROOT, "tiramisu_amd", "programs")
SMALL = [(128, 192, 128), (48, 40, 24), (200, 150, 100), (1024, 1280, 512)]
RTOL = 2e-2


def to_bf16(a):
    """fp32 -> bf16 bits, round to nearest even (the storage format of p_bfloat16 buffers)."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = 0x7FFF + ((u >> 16) & 1)
    return ((u + r) >> 16).astype(np.uint16)


def from_bf16(b):
    return (b.astype(np.uint32) << 16).view(np.float32)


def name_of(M, N, K):
    return "sgemm_bf16_%dx%dx%d" % (M, N, K)


def cpu_program(M, N, K):
    n = name_of(M, N, K)
    return runtime.Program(oracle_build.cpu_program_library(PROGRAMS, n), n, needs_gpu_runtime=False)


def test_bf16_rounding_helper():
    # exactly representable values survive; ties go to even
    x = np.array([1.0, -2.5, 0.15625, 3.0e38], np.float32)
    assert np.array_equal(from_bf16(to_bf16(x))[:3], x[:3])
    tie = np.array([0x3F808000], np.uint32).view(np.float32)      # 1.00390625: halfway between two bf16
    assert to_bf16(tie)[0] == 0x3F80
    tie2 = np.array([0x3F818000], np.uint32).view(np.float32)
    assert to_bf16(tie2)[0] == 0x3F82


@pytest.mark.parametrize("M,N,K,what", [(128, 192, 128, "tile 64x64x64, whole tiles"), (48, 40, 24, "tile 64x64x64, guarded edges"),
                                        (200, 150, 100, "tile 64x64x64, guarded edges"), (1024, 1280, 512, "tile 128x128x32, whole tiles"),
                                        (4096, 4096, 4096, "tile 256x256x32, whole tiles")])
def test_every_shape_gets_the_bf16_mfma_kernel(M, N, K, what):
    """Ragged shapes and unaligned rows take the 64x64 tile with guarded loads instead of falling back
    to the schedule-faithful (VALU) kernel."""
    import json
    kernels = json.load(open(os.path.join(PROGRAMS, "build", name_of(M, N, K) + ".o.json")))["kernels"]
    assert len(kernels) == 1 and "v_mfma_f32_32x32x16_bf16" in kernels[0]["how"] and what in kernels[0]["how"]


@pytest.mark.parametrize("M,N,K", [(640, 704, 64), (70, 66, 130), (2000, 1500, 1006)])
def test_loads_of_the_epilogue_are_in_flight_together(M, N, K, programs_dir, tmp_path):
    """In the instructions of the kernel, the loads of C are not waited for one by one, each before the next is issued."""
    import subprocess
    from tiramisu_amd import build
    text = str(tmp_path / "kernel.s")
    subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["--cuda-device-only", "-S", "-I" + os.path.join(build.CSRC, "kernels"), "-o", text,
                    os.path.join(programs_dir, "build", name_of(M, N, K) + ".o.hip")], check=True, stderr=subprocess.DEVNULL)
    loads, alone, last = 0, 0, ""
    for line in open(text):
        words = line.split()
        if words[:1] == ["s_endpgm"]:
            break                               # of the kernel for operands at multiples of four bytes
        if words and words[0] in ("global_load_dword", "global_store_dword"):
            loads += words[0] == "global_load_dword"
            last = words[0]
        elif words[:2] == ["s_waitcnt", "vmcnt(0)"]:
            alone += last == "global_load_dword"
            last = ""
    assert loads >= 16 and alone <= loads // 8, "%d of %d loads waited for one by one" % (alone, loads)


@pytest.mark.parametrize("M,N,K", SMALL)
def test_cpu_generated_code_matches_float64(M, N, K):
    rng = np.random.RandomState(M + K)
    A, B = to_bf16(rng.uniform(-1, 1, (M, K))), to_bf16(rng.uniform(-1, 1, (K, N)))
    C = rng.uniform(-1, 1, (M, N)).astype(np.float32)
    exact = 1.5 * (from_bf16(A).astype(np.float64) @ from_bf16(B).astype(np.float64)) + 0.5 * C
    cpu_program(M, N, K)(np.array([1.5, 0.5], np.float32), A, B, C)
    assert np.max(np.abs(C - exact)) <= 1e-5 * np.max(np.abs(exact))


def run_gpu(M, N, K, scal, A, B, C):
    from gpu_util import DeviceArray
    d = [DeviceArray(a) for a in (A, B, C)]
    runtime.load(PROGRAMS, name_of(M, N, K))(scal, *[x.buffer() for x in d])
    out = d[2].download()
    for x in d:
        x.free()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SMALL)
def test_gpu_matches_cpu_generated_code(M, N, K):
    rng = np.random.RandomState(2 * M + K)
    scal = np.array([1.0, 0.0], np.float32)
    # integer-valued data: exact on every path
    A, B = to_bf16(rng.randint(-5, 5, (M, K)).astype(np.float32)), to_bf16(rng.randint(-5, 5, (K, N)).astype(np.float32))
    C = np.zeros((M, N), np.float32)
    C_cpu = C.copy()
    cpu_program(M, N, K)(scal, A, B, C_cpu)
    assert np.array_equal(run_gpu(M, N, K, scal, A, B, C), C_cpu)
    # uniform data
    A, B = to_bf16(rng.uniform(-1, 1, (M, K))), to_bf16(rng.uniform(-1, 1, (K, N)))
    cpu_program(M, N, K)(scal, A, B, C_cpu)
    out = run_gpu(M, N, K, scal, A, B, C)
    from gpu_util import assert_fp32_parity
    assert_fp32_parity(out, C_cpu, "sgemm bf16 vs CPU-generated code", RTOL)


@pytest.mark.gpu
def test_gpu_4096_sampled_rows():
    M = N = K = 4096
    rng = np.random.RandomState(40)
    scal = np.array([1.0, 0.0], np.float32)
    A, B = to_bf16(rng.uniform(-1, 1, (M, K))), to_bf16(rng.uniform(-1, 1, (K, N)))
    out = run_gpu(M, N, K, scal, A, B, np.zeros((M, N), np.float32))
    rows = rng.choice(M, 32, replace=False)
    exact = from_bf16(A[rows]).astype(np.float64) @ from_bf16(B).astype(np.float64)
    from gpu_util import assert_fp32_parity
    assert_fp32_parity(out[rows], exact, "sgemm bf16 4096^3 sampled rows vs float64", RTOL)
    # integer-valued data: exact
    A, B = to_bf16(rng.randint(-3, 4, (M, K)).astype(np.float32)), to_bf16(rng.randint(-3, 4, (K, N)).astype(np.float32))
    out = run_gpu(M, N, K, scal, A, B, np.zeros((M, N), np.float32))
    exact = from_bf16(A[rows]).astype(np.float64) @ from_bf16(B).astype(np.float64)
    assert np.array_equal(out[rows], exact.astype(np.float32))


def how(directory, name):
    import json
    return json.load(open(os.path.join(directory, "build", name + ".o.json")))["kernels"][0]["how"]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4096, 3072, 32), (3072, 4096, 160)])
def test_gpu_large_tiles_short_k(M, N, K):
    """128x128 tiles (slices loaded straight into the four-stage LDS ring) with one and five K-slices:
    the ring's start-up, a single steady-state turn and the drain, every element checked, with the
    alpha / beta epilogue."""
    assert "straight into LDS" in how(PROGRAMS, name_of(M, N, K)) and "tile 128x128x32, whole tiles" in how(PROGRAMS, name_of(M, N, K))
    rng = np.random.RandomState(M + K)
    scal = np.array([1.5, 0.5], np.float32)
    A, B = to_bf16(rng.randint(-4, 5, (M, K)).astype(np.float32)), to_bf16(rng.randint(-4, 5, (K, N)).astype(np.float32))
    C = rng.randint(-8, 9, (M, N)).astype(np.float32)
    exact = 1.5 * (from_bf16(A).astype(np.float64) @ from_bf16(B).astype(np.float64)) + 0.5 * C
    assert np.array_equal(run_gpu(M, N, K, scal, A, B, C.copy()), exact.astype(np.float32))     # integer data: exact
    A, B = to_bf16(rng.uniform(-1, 1, (M, K))), to_bf16(rng.uniform(-1, 1, (K, N)))
    exact = 1.5 * (from_bf16(A).astype(np.float64) @ from_bf16(B).astype(np.float64)) + 0.5 * C
    out = run_gpu(M, N, K, scal, A, B, C.copy())
    assert np.max(np.abs(out - exact)) <= 1e-5 * np.max(np.abs(exact))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(20480, 20480, 32), (8192, 12288, 96), (8192, 8192, 160)])
def test_gpu_largest_tiles_short_k(M, N, K, programs_dir):
    """256x256 tiles, which the model takes for large planes where K is short, with one, three and five K-slices of the four-stage
    ring: every element against torch's fp32 product, exact for small integers."""
    import torch
    name = name_of(M, N, K)
    assert "straight into LDS" in how(programs_dir, name) and "tile 256x256x32, whole tiles" in how(programs_dir, name)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K)
    A, B = (torch.randint(-4, 5, s, generator=g, device="cuda").float() for s in ((M, K), (K, N)))
    C = torch.randint(-8, 9, (M, N), generator=g, device="cuda", dtype=torch.int8).float()
    exact = torch.addmm(C, A, B, beta=0.5, alpha=2.0)
    runtime.load(programs_dir, name)(np.array([2.0, 0.5], np.float32), A.to(torch.bfloat16), B.to(torch.bfloat16), C)
    assert torch.equal(C, exact)
    del A, B, C, exact
    torch.cuda.empty_cache()


EDGES = [(4002, 3998, 500, "tile 256x256x32, guarded edges"), (2000, 1500, 1006, "tile 128x128x32, guarded edges"),
         (70, 66, 130, "tile 64x64x64, guarded edges"), (66, 2, 6, "tile 64x64x64, guarded edges"),
         (2001, 1501, 1001, "tile 128x128x64, guarded edges"), (65, 67, 193, "tile 64x64x64, guarded edges"),
         (64, 65, 63, "tile 64x64x64, guarded edges"), (33, 3, 65, "tile 64x64x64, guarded edges")]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,what", EDGES)
def test_gpu_sizes_that_end_inside_a_tile(M, N, K, what, programs_dir):
    """Small integers: every sum is exact.  First all finite, so that every element counts; then with the first elements of A's
    even rows, of its odd ones, and of every other row of B infinite: a row read past its end goes on into the next one's, which
    must not be used (where they belong, they make a row or the first column of the result infinite)."""
    from gpu_util import DeviceArray
    tile = how(programs_dir, name_of(M, N, K))
    assert what in tile and ("straight into LDS" in tile) == (K % 2 == 0 and N % 2 == 0)
    rng = np.random.RandomState(M + N + K)
    for infinite in ("nothing", "even rows of A", "odd rows of A", "rows of B"):
        A, B = rng.randint(-3, 4, (M, K)).astype(np.float32), rng.randint(1, 4, (K, N)).astype(np.float32)
        if infinite.endswith("A"):
            A[infinite.startswith("odd")::2, 0] = np.inf
        elif infinite.endswith("B"):
            B[1::2, 0] = np.inf
        C = rng.randint(-8, 9, (M, N)).astype(np.float32)
        with np.errstate(invalid="ignore"):
            exact = 2.0 * (A @ B) + 0.5 * C        # sums of at most 1006 products below 10: exact in float32 in any order
        d = [DeviceArray(a) for a in (to_bf16(A), to_bf16(B), C)]
        runtime.load(programs_dir, name_of(M, N, K))(np.array([2.0, 0.5], np.float32), *[x.buffer() for x in d])
        assert np.array_equal(d[2].download(), exact, equal_nan=True), infinite


TILES = [(1793, 3842, 514, "tile 128x256x64, guarded edges"), (1921, 2562, 578, "tile 192x128x64, guarded edges"),
         (673, 3202, 1090, "tile 96x128x64, guarded edges"), (1473, 642, 514, "tile 64x128x64, guarded edges"), (33, 66, 194, "tile 32x64x64, guarded edges"),
         (2000, 1500, 1010, "tile 128x128x32, guarded edges, slices in pairs"), (3842, 3970, 1278, "tile 256x256x32, guarded edges, slices in pairs"),
         (1920, 2560, 1024, "tile 192x128x64, whole tiles"),
         # 192 tiles of 256 and rows of A at whole lines: pairs; 140 tiles: one by one; rows at 16 bytes: 128 x 128 rather than two rounds of 192 x 128
         (3841, 3074, 1088, "tile 256x256x32, guarded edges, slices in pairs"), (2560, 3520, 1368, "tile 256x256x32, guarded edges, 1 product"),
         (4096, 2560, 640, "tile 128x128x32, whole tiles, 1 product")]


@pytest.mark.parametrize("M,N,K,what", TILES)
def test_tiles_of_the_model(M, N, K, what, programs_dir):
    assert what in how(programs_dir, name_of(M, N, K))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,what", TILES)
def test_gpu_tiles_between_the_squares(M, N, K, what, programs_dir):
    """The tiles between the squares of 256, 128 and 64, and slices in pairs or one by one, at their remainders: exact as above."""
    test_gpu_sizes_that_end_inside_a_tile(M, N, K, what, programs_dir)


VIEWS = [("a_backwards", 200, 150, 100), ("b_backwards", 200, 150, 100), ("a_backwards_whole", 128, 192, 128), ("b_backwards_whole", 128, 192, 128),
         ("b_overlapping", 66, 30, 50)]


@pytest.mark.parametrize("form", [v[0] for v in VIEWS])
def test_operands_walked_backwards_or_overlapping_are_not_loaded_straight_into_lds(form, programs_dir):
    """Those loads address an operand by 32-bit offsets from its first row and rely on what follows its last row reading as zero."""
    tile = how(programs_dir, "sgemm_bf16_" + form)
    assert "v_mfma_f32_32x32x16_bf16" in tile and "straight into LDS" not in tile


@pytest.mark.gpu
@pytest.mark.parametrize("form,M,N,K", VIEWS)
def test_gpu_operands_walked_backwards_or_overlapping(form, M, N, K, programs_dir):
    from gpu_util import DeviceArray
    rng = np.random.RandomState(M + N + K)
    A, B = rng.randint(-3, 4, (M, K)).astype(np.float32), rng.randint(-3, 4, (K, N)).astype(np.float32)
    C = rng.randint(-8, 9, (M, N)).astype(np.float32)
    stored_a, stored_b = A, B
    if form.startswith("a_"):
        stored_a = A[::-1]
    elif form != "b_overlapping":
        stored_b = B[::-1]
    else:                                       # row k begins at element 2 k: what lies behind the last row must not be used
        stored_b = np.full((K, N + 2 * K), np.inf, np.float32)
        stored_b[0, :2 * (K - 1) + N] = rng.randint(-3, 4, 2 * (K - 1) + N)
        B = np.stack([stored_b[0, 2 * k:2 * k + N] for k in range(K)])
    d = [DeviceArray(a) for a in (to_bf16(stored_a), to_bf16(stored_b), C)]
    runtime.load(programs_dir, "sgemm_bf16_" + form)(*[x.buffer() for x in d])
    assert np.array_equal(d[2].download(), A @ B + C)       # integers: exact


@pytest.mark.gpu
@pytest.mark.parametrize("form,M,N,K,lda,ldb", [("odd_k", 200, 150, 101, 102, 150), ("odd_n", 200, 149, 100, 100, 150),
                                                ("odd_k_and_n", 129, 257, 33, 36, 258)])
def test_gpu_odd_parts_of_rows_of_an_even_number_of_elements(form, M, N, K, lda, ldb, programs_dir):
    """The last element of the last row is the first half of a dword whose second half is not part of the operand."""
    from gpu_util import DeviceArray
    assert "straight into LDS" in how(programs_dir, "sgemm_bf16_" + form)
    rng = np.random.RandomState(M + N + K)
    A, B = np.full((M, lda), np.inf, np.float32), np.full((K, ldb), np.inf, np.float32)
    A[:, :K], B[:, :N] = rng.randint(1, 4, (M, K)), rng.randint(1, 4, (K, N))        # no zeros: a lost element shows
    C = rng.randint(-8, 9, (M, N)).astype(np.float32)
    d = [DeviceArray(a) for a in (to_bf16(A), to_bf16(B), C)]
    runtime.load(programs_dir, "sgemm_bf16_" + form)(*[x.buffer() for x in d])
    assert np.array_equal(d[2].download(), A[:, :K] @ B[:, :N] + C)       # integers: exact


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(200, 150, 100), (128, 192, 128), (1024, 1280, 512), (2000, 1500, 1006), (66, 2, 6)])
@pytest.mark.parametrize("odd_a,odd_b", [(True, False), (False, True), (True, True)])
def test_gpu_operands_that_begin_at_an_odd_element(M, N, K, odd_a, odd_b, programs_dir):
    """Contiguous parts of larger tensors: the loads straight into LDS want multiples of four bytes, so another kernel serves
    these addresses.  Infinities around the operands must not be used."""
    import torch
    rng = np.random.RandomState(M + N + K)

    def part(rows, cols, odd):
        flat = torch.full((rows * cols + 9,), float("inf"), dtype=torch.bfloat16)
        values = rng.randint(-3, 4, (rows, cols)).astype(np.float32)
        first = 7 if odd else 4
        flat[first:first + rows * cols] = torch.from_numpy(values).flatten()
        view = flat.cuda()[first:first + rows * cols].view(rows, cols)
        assert view.data_ptr() % 4 == (2 if odd else 0)
        return view, values

    (dA, A), (dB, B) = part(M, K, odd_a), part(K, N, odd_b)
    C = rng.randint(-8, 9, (M, N)).astype(np.float32)
    dC = torch.from_numpy(C).cuda()
    directory = PROGRAMS if os.path.exists(os.path.join(PROGRAMS, "build", name_of(M, N, K) + ".o.json")) else programs_dir
    runtime.load(directory, name_of(M, N, K))(np.array([2.0, 0.5], np.float32), dA, dB, dC)
    assert np.array_equal(dC.cpu().numpy(), 2.0 * (A @ B) + 0.5 * C)       # sums of at most 1006 products up to 9: exact in float32
