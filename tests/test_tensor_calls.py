"""Calls whose arguments are all GPU tensors go through one entry of the runtime (tiramisu_hip_call); everything else takes the general way and
is refused as before."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tiramisu_amd import runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAMS = os.path.join(ROOT, "tiramisu_amd", "programs")


def test_the_function_sees_the_buffers_that_the_general_way_describes(tmp_path):
    """Without a GPU: functions of one to eight arguments write down what they are given, on a stream that is only passed on."""
    names = ["b%d" % i for i in range(8)]
    (tmp_path / "f.cpp").write_text("""#include <stdint.h>
struct dim { int32_t min, extent, stride; uint32_t flags; };
struct buf { uint64_t device; void *iface; uint8_t *host; uint64_t flags; uint8_t code, bits; uint16_t lanes; int32_t nd; dim *d; void *pad; };
int64_t seen[8][40];
static int note(buf **b, int n) {
    for (int i = 0; i < n; i++) {
        int64_t *s = seen[i];
        *s++ = b[i]->device; *s++ = (int64_t)b[i]->iface + (int64_t)b[i]->host + b[i]->flags; *s++ = b[i]->code; *s++ = b[i]->bits; *s++ = b[i]->lanes; *s++ = b[i]->nd;
        for (int d = 0; d < b[i]->nd; d++) { *s++ = b[i]->d[d].min; *s++ = b[i]->d[d].extent; *s++ = b[i]->d[d].stride; *s++ = b[i]->d[d].flags; }
    }
    return 10 + n;
}
""" + "".join('extern "C" int f%d(%s) { buf *b[] = {%s}; return note(b, %d); }\n' % (n, ", ".join("buf *" + v for v in names[:n]), ", ".join(names[:n]), n)
              for n in range(1, 9)))
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "f.so"), str(tmp_path / "f.cpp")], check=True)
    lib, w = ctypes.CDLL(str(tmp_path / "f.so")), runtime.wrappers()
    shapes, types = [(3,), (4, 5), (2, 3, 4), (7, 1), (6, 2, 2, 3), (9,), (1,), (2, 8)], [(2, 32), (2, 64), (0, 32), (1, 16), (2, 32), (0, 8), (1, 64), (2, 32)]
    before = w.tiramisu_hip_get_stream()
    for n in range(1, 10):
        count = min(n, 8)
        text = []
        for s, t in zip(shapes[:count], types):
            text += [t[0], t[1], len(s)] + list(s)
        pointers = (ctypes.c_uint64 * 9)(*[1000 + i for i in range(9)])
        f = getattr(lib, "f%d" % count)
        rc = w.tiramisu_hip_call(ctypes.cast(f, ctypes.c_void_p), n, pointers, (ctypes.c_int32 * len(text))(*text), ctypes.c_void_p(4096))
        assert rc == (10 + n if n <= 8 else -1) and w.tiramisu_hip_get_stream() == before
    seen = ((ctypes.c_int64 * 40) * 8).in_dll(lib, "seen")
    for i, (s, (code, bits)) in enumerate(zip(shapes, types)):
        b = runtime.Buffer.from_device(1000 + i, s, {(2, 32): "f4", (2, 64): "f8", (0, 32): "i4", (1, 16): "u2", (0, 8): "i1", (1, 64): "u8"}[code, bits])
        general = [b.raw.device, 0, b.raw.type.code, b.raw.type.bits, b.raw.type.lanes, b.raw.dimensions]
        for d in range(b.raw.dimensions):
            general += [b.dims[d].min, b.dims[d].extent, b.dims[d].stride, b.dims[d].flags]
        assert list(seen[i])[:len(general)] == general


def test_which_functions_take_tensors_only():
    conv, product = runtime.load(PROGRAMS, "conv2d_2x8x64x16"), runtime.load(PROGRAMS, "sgemm_128x192x96")
    assert [s for _, s in conv.of_tensors[2]] == [(2, 8, 18, 18), (64, 8, 3, 3), (64,), (2, 64, 16, 16)]
    assert product.of_tensors is None                    # its two scalars are a host buffer


@pytest.mark.gpu
def test_tensor_calls_on_the_default_and_a_side_stream_and_what_is_refused():
    import torch
    p, w = runtime.load(PROGRAMS, "conv2d_2x8x64x16"), runtime.wrappers()
    g = torch.Generator().manual_seed(1)
    x, weights, bias = (torch.randint(-3, 4, s, generator=g).float().cuda() for s in ((2, 8, 18, 18), (64, 8, 3, 3), (64,)))
    expected = torch.relu(torch.nn.functional.conv2d(x.cpu().double(), weights.cpu().double(), bias.cpu().double()))
    out = torch.zeros(2, 64, 16, 16, device="cuda")
    runtime.Buffer.from_tensor(out)                      # (torch's types are known)
    before, calls, one_entry = w.tiramisu_hip_get_stream(), [], p._call_of_tensors
    p._call_of_tensors = lambda args: calls.append(one_entry(args)) or calls[-1]
    p(x, weights, bias, out)
    assert calls == [0] and torch.equal(out.cpu().double(), expected)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        twice = x * 2.0                                  # made on the side stream just before the call
        out2 = torch.zeros_like(out)
        p(twice, weights, bias, out2)
        result = out2 + 0.0
    side.synchronize()
    assert calls == [0, 0] and w.tiramisu_hip_get_stream() == before
    assert torch.equal(result.cpu().double(), torch.relu(torch.nn.functional.conv2d(2 * x.cpu().double(), weights.cpu().double(), bias.cpu().double())))
    # another shape with as many elements takes the general way, and so does a part of a larger tensor that begins anywhere
    p(x, weights.reshape(64, 72), bias, out.zero_())
    assert calls[-1] is None and torch.equal(out.cpu().double(), expected)
    part = torch.cat([torch.full((1,), float("nan"), device="cuda"), x.flatten()])[1:].view(x.shape)
    p(part, weights, bias, out.zero_())
    assert calls[-1] == 0 and torch.equal(out.cpu().double(), expected)
    for wrong in ((x.cpu(), weights, bias, out), (x.double(), weights, bias, out), (x[:1], weights, bias, out), (x, weights, bias)):
        with pytest.raises(ValueError):
            p(*wrong)
        assert calls[-1] is None
    with pytest.raises(ValueError):
        p(x.transpose(2, 3), weights, bias, out)
    p._call_of_tensors, seen, fn = one_entry, [], p.fn
    p.fn = lambda *a: (seen.append(len(a)), fn(*a))[1]   # a caller's own function in its place is called
    p(x, weights, bias, out.zero_())
    assert seen == [4] and torch.equal(out.cpu().double(), expected)


@pytest.mark.gpu
def test_weights_held_as_parameters_take_the_one_entry():
    import torch
    p = runtime.load(PROGRAMS, "conv2d_2x8x64x16")
    x, out = torch.ones(2, 8, 18, 18, device="cuda"), torch.zeros(2, 64, 16, 16, device="cuda")
    layer = torch.nn.Conv2d(8, 64, 3).cuda()
    with torch.no_grad():
        layer.weight.fill_(0.25)
        layer.bias.fill_(1.0)
    calls, one_entry = [], p._call_of_tensors
    p._call_of_tensors = lambda args: calls.append(one_entry(args)) or calls[-1]
    p(x, layer.weight, layer.bias, out)
    assert calls == [0] and torch.all(out == 8 * 9 * 0.25 + 1.0)


@pytest.mark.gpu
def test_tensor_calls_follow_torch_work_in_two_threads():
    import threading
    import torch
    p = runtime.load(PROGRAMS, "conv2d_2x8x64x16")
    weights, bias = torch.zeros(64, 8, 3, 3, device="cuda"), torch.zeros(64, device="cuda")
    weights[:, 0, 1, 1] = 1.0
    big, failed = torch.zeros(2048, 2048, device="cuda"), []

    def repeat(first):
        try:
            for i in range(first, first + 5):
                x, out = torch.zeros(2, 8, 18, 18, device="cuda"), torch.zeros(2, 64, 16, 16, device="cuda")
                y = big
                for _ in range(10):                      # torch work in flight, then the input
                    y = y @ big
                x += y[0, 0] + float(i + 1)
                p(x, weights, bias, out)
                assert torch.all(out * 1.0 == i + 1)
        except BaseException as e:
            failed.append(e)

    repeat(0)
    threads = [threading.Thread(target=repeat, args=(10 * t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
