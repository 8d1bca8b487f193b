"""The workloads whose speed this framework is judged by, as a program of its user runs them.

A case names a kind of work and its sizes.  Five kinds are Tiramisu programs of tiramisu_amd/programs, compiled for the sizes
and called through runtime.Program: sgemm, sgemm_bf16, conv2d, lstm, heat2d.  A size that the build already made is loaded; any
other is generated on first use, as a user who writes the program for it does, and kept in a temporary directory of this user.
Two kinds are the GEMM library calls that cublas_gemm() in a program leads to (tiramisu_hip_sgemm, tiramisu_hip_dgemm), whose
sizes are run-time values.  All tensors live on the GPU: the programs take GPU-resident arguments.
"""
import hashlib
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from tiramisu_amd import build, runtime

PROGRAMS = os.path.join(build.PKG, "programs")


def listed():
    return [
        # benchmark configuration: one C tile per compute unit, a single short launch
        {"name": "sgemm 1024", "kind": "sgemm", "M": 1024, "N": 1024, "K": 1024},
        # benchmark configuration: the large fp32 product
        {"name": "sgemm 4096", "kind": "sgemm", "M": 4096, "N": 4096, "K": 4096},
        # a run-time sized call with a transposed operand, no dimension a multiple of a tile
        {"name": "sgemm call, A transposed", "kind": "sgemm_call", "M": 1000, "N": 1500, "K": 700, "tA": True, "tB": False},
        # double precision, ragged in M, N and K, B transposed, C updated
        {"name": "dgemm call, B transposed", "kind": "dgemm_call", "M": 1500, "N": 1430, "K": 250, "tA": False, "tB": True},
        # benchmark configuration: bf16 inputs, fp32 accumulation
        {"name": "sgemm bf16 4096", "kind": "sgemm_bf16", "M": 4096, "N": 4096, "K": 4096},
        # the same program at a size that no tile divides
        {"name": "sgemm bf16 ragged", "kind": "sgemm_bf16", "M": 2000, "N": 1500, "K": 1000},
        # benchmark configuration: a middle layer of a convolutional network
        {"name": "conv2d 64 to 64", "kind": "conv2d", "N": 32, "CI": 64, "CO": 64, "H": 112},
        # its first layer: three colour channels
        {"name": "conv2d 3 to 64", "kind": "conv2d", "N": 8, "CI": 3, "CO": 64, "H": 112},
        # benchmark configuration: a long sequence through a stack of layers
        {"name": "lstm 4x64x512x100", "kind": "lstm", "L": 4, "B": 64, "H": 512, "S": 100},
        # a small network and a short sequence: latency and launches
        {"name": "lstm 3x20x64x4", "kind": "lstm", "L": 3, "B": 20, "H": 64, "S": 4},
        # benchmark configuration: a plane of 256 MiB
        {"name": "heat2d 8192x32", "kind": "heat2d", "N": 8192, "STEPS": 32},
        # a small plane whose rows are not a multiple of 16 bytes
        {"name": "heat2d 1030x9", "kind": "heat2d", "N": 1030, "STEPS": 9},
    ]


def draw(rng):
    def size(low, high, step=1):
        """Spread over the logarithm; half of the sizes are what they are, half a multiple of `step`."""
        v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
        if step > 1 and rng.random() < 0.5:
            v = (v + step // 2) // step * step
        return max(low, min(high, v))

    kind = rng.choice(["sgemm", "sgemm_bf16", "sgemm_call", "dgemm_call", "conv2d", "lstm", "heat2d"])
    if kind in ("sgemm", "sgemm_bf16"):
        return {"kind": kind, "M": size(32, 4096, 64), "N": size(32, 4096, 64), "K": size(32, 4096, 64)}
    if kind in ("sgemm_call", "dgemm_call"):
        top = 4096 if kind == "sgemm_call" else 2048
        return {"kind": kind, "M": size(16, top, 32), "N": size(16, top, 32), "K": size(16, top, 32),
                "tA": rng.random() < 0.5, "tB": rng.random() < 0.5}
    if kind == "conv2d":
        return {"kind": kind, "N": size(1, 32), "CI": size(3, 64, 8), "CO": size(5, 64, 16), "H": size(8, 112, 8)}
    if kind == "lstm":
        return {"kind": kind, "L": rng.randint(1, 4), "B": size(4, 64, 8), "H": size(16, 512, 32), "S": size(3, 100)}
    return {"kind": kind, "N": size(20, 8192, 64), "STEPS": size(2, 32)}


# ---------------------------------------------------------------- compiled programs

_SIZES = {"sgemm": ("M", "N", "K"), "sgemm_bf16": ("M", "N", "K"), "conv2d": ("N", "CI", "CO", "H"), "lstm": ("L", "B", "H", "S"),
          "heat2d": ("N", "STEPS")}


def _compiler_version():
    """What generated code depends on: the compiler library and the kernel headers it includes."""
    h = hashlib.sha1(open(build.compiler_library(), "rb").read())
    kernels = os.path.join(build.CSRC, "kernels")
    for f in sorted(os.listdir(kernels)):
        h.update(open(os.path.join(kernels, f), "rb").read())
    return h.hexdigest()[:16]


def _program(case):
    """The compiled function for the case's sizes."""
    kind, sizes = case["kind"], [case[k] for k in _SIZES[case["kind"]]]
    name = kind + "_" + "x".join(str(v) for v in sizes)
    if os.path.exists(build.program_library(PROGRAMS, name)):
        return runtime.load(PROGRAMS, name)
    keep = os.path.join(tempfile.gettempdir(), "tiramisu_programs_%d" % os.getuid(),
                        hashlib.sha1(build.PKG.encode()).hexdigest()[:8] + "_" + _compiler_version())
    directory = os.path.join(keep, name)
    if not os.path.exists(build.program_library(directory, name)):
        os.makedirs(keep, exist_ok=True)
        work = tempfile.mkdtemp(prefix=name + ".", dir=keep)
        source = os.path.join(work, name + ".cpp")
        with open(source, "w") as f:
            f.write('#define main main_of_all_sizes\n#include "%s"\n#undef main\nint main() { generate(%s); return 0; }\n'
                    % (os.path.join(PROGRAMS, kind + ".cpp"), ", ".join(str(v) for v in sizes)))
        os.environ["TIRAMISU_AMD_KERNEL_DIR"] = os.path.join(build.CSRC, "kernels")
        os.environ["TIRAMISU_AMD_INCLUDE"] = build.INCLUDE
        build.build_program(source, directory=work)
        try:
            os.rename(work, directory)
        except OSError:                      # another process was first
            shutil.rmtree(work, ignore_errors=True)
    return runtime.load(directory, name)


# ---------------------------------------------------------------- inputs and passes

def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def uniform(shape, low, high, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda").uniform_(low, high, generator=g)

    if kind in ("sgemm", "sgemm_bf16"):
        M, N, K = case["M"], case["N"], case["K"]
        A, B, C = uniform((M, K), -1, 1), uniform((K, N), -1, 1), torch.zeros((M, N), device="cuda")
        if kind == "sgemm_bf16":
            A, B = A.to(torch.bfloat16), B.to(torch.bfloat16)
        scal = np.array([1.0, 0.0], np.float32)
        buffers = [runtime.Buffer.from_numpy(scal)] + [runtime.Buffer.from_tensor(t) for t in (A, B, C)]
        return {"call": _program(case), "arguments": buffers, "out": C}
    if kind in ("sgemm_call", "dgemm_call"):
        M, N, K, tA, tB = (case[k] for k in ("M", "N", "K", "tA", "tB"))
        dtype = torch.float32 if kind == "sgemm_call" else torch.float64
        A = uniform((K, M) if tA else (M, K), -1, 1, dtype)
        B = uniform((N, K) if tB else (K, N), -1, 1, dtype)
        C = uniform((M, N), -1, 1, dtype)
        w = runtime.wrappers()
        call, alpha, beta = (w.tiramisu_hip_sgemm, 1.0, 0.0) if kind == "sgemm_call" else (w.tiramisu_hip_dgemm, 1.5, 0.5)
        return {"call": call, "arguments": [A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, alpha, beta, 0, 0, 0, 0, 0, 0, tA, tB],
                "tensors": (A, B), "out": C}
    if kind == "conv2d":
        NB, CI, CO, H = case["N"], case["CI"], case["CO"], case["H"]
        padded = torch.zeros((NB, CI, H + 2, H + 2), device="cuda")
        padded[:, :, 1:-1, 1:-1] = uniform((NB, CI, H, H), 0, 1)
        w, bias = uniform((CO, CI, 3, 3), -0.1, 0.1), uniform((CO,), -0.1, 0.1)
        out = torch.zeros((NB, CO, H, H), device="cuda")
        return {"call": _program(case), "arguments": [padded, w, bias, out], "out": out}
    if kind == "lstm":
        L, B, H, S = case["L"], case["B"], case["H"], case["S"]
        weights, biases = uniform((L, 2, 4 * H, H), -0.08, 0.08), uniform((L, 4 * H), -0.08, 0.08)
        x, y = uniform((S, B, H), -1, 1), torch.zeros((S, B, H), device="cuda")
        return {"call": _program(case), "arguments": [weights, biases, x, y], "out": y}
    planes = uniform((2, case["N"], case["N"]), 0, 1)
    planes[1] = planes[0]                    # the boundary is fixed: both planes hold it
    return {"call": _program(case), "arguments": [runtime.Buffer.from_tensor(planes)], "out": planes}


def run(state):
    state["call"](*state["arguments"])
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("sgemm", "sgemm_bf16", "sgemm_call", "dgemm_call"):
        M, N, K = case["M"], case["N"], case["K"]
        inputs, result = {"sgemm": (4, 4), "sgemm_bf16": (2, 4), "sgemm_call": (4, 4), "dgemm_call": (8, 8)}[kind]
        # C is read where the scaling of it is not zero, or where the program says C * beta
        passes_over_c = 1 if kind == "sgemm_call" else 2
        return {"bytes": inputs * (M * K + K * N) + passes_over_c * result * M * N, "flops": 2 * M * N * K}
    if kind == "conv2d":
        NB, CI, CO, H = case["N"], case["CI"], case["CO"], case["H"]
        return {"bytes": 4 * (NB * CI * (H + 2) ** 2 + CO * CI * 9 + CO + NB * CO * H * H), "flops": 2 * NB * CO * H * H * CI * 9}
    if kind == "lstm":
        L, B, H, S = case["L"], case["B"], case["H"], case["S"]
        return {"bytes": 4 * (L * 8 * H * H + L * 4 * H + 2 * S * B * H), "flops": L * S * 2 * (2 * B * 4 * H * H)}
    N, steps = case["N"], case["STEPS"]
    # one plane read, both planes written: the last step and the last but one
    return {"bytes": 4 * 3 * N * N, "flops": 5 * (N - 2) ** 2 * steps}


def tolerance(case):
    # four times the distance from the same path in 64 bits, at the sizes listed and at drawn ones: products of up to 4096 terms
    # 1.2e-6 in fp32 and 4e-7 with bf16 inputs (exact products), convolutions 5e-7, a hundred LSTM steps 3e-7, 32 stencil steps
    # 7e-7; the double precision product is off from another order of its sums by 6e-16 at 250 terms, and at most 2e-15 at 2048
    return {"rel": {"sgemm": 5e-6, "sgemm_call": 5e-6, "dgemm_call": 1e-14, "sgemm_bf16": 2e-6, "conv2d": 2e-6, "lstm": 1.5e-6,
                    "heat2d": 3e-6}[case["kind"]]}
