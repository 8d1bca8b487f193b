"""Calling compiled Tiramisu functions from Python through their C ABI.

A compiled Tiramisu function is ``extern "C" int f(halide_buffer_t *arg0, ...)``
(reference: the generated headers, e.g. tests/wrapper_test_167.h, and the buffer layout at
benchmarks/linear_algebra/blas/level1/dot/generated_dot.o.h:1157-1219).  This module is the
Python counterpart of the reference's C++ wrapper programs: it describes numpy arrays (host
memory) or raw device pointers as ``halide_buffer_t`` and calls the function with ctypes.
It contains no compute of its own and has no CPU fallback: loading fails loudly when the
HIP libraries were not built.
"""
import ctypes
import functools
import math
import os
import struct
import sys

import numpy as np

from . import build as _build


class halide_dimension_t(ctypes.Structure):
    _fields_ = [("min", ctypes.c_int32), ("extent", ctypes.c_int32), ("stride", ctypes.c_int32),
                ("flags", ctypes.c_uint32)]


class halide_type_t(ctypes.Structure):
    _fields_ = [("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16)]


class halide_buffer_t(ctypes.Structure):
    _fields_ = [("device", ctypes.c_uint64), ("device_interface", ctypes.c_void_p),
                ("host", ctypes.c_void_p), ("flags", ctypes.c_uint64), ("type", halide_type_t),
                ("dimensions", ctypes.c_int32), ("dim", ctypes.POINTER(halide_dimension_t)),
                ("padding", ctypes.c_void_p)]


_TYPE_CODES = {"i": 0, "u": 1, "f": 2, "b": 1}
_DIMENSIONS_OF = ctypes.POINTER(halide_dimension_t)
_tensor_types = {}                                            # torch's element types as numpy's


def _tensor_type(t):
    if t not in _tensor_types:
        import torch
        _tensor_types[t] = np.dtype(np.uint16) if t == torch.bfloat16 else np.dtype(str(t).replace("torch.", ""))
    return _tensor_types[t]


class Buffer:
    """Owns the ``halide_buffer_t`` (and its dimension array) describing one argument.

    Dimensions are stored innermost first, as Halide does: a C-contiguous numpy array of shape
    (M, N) has dim[0] = N (stride 1) and dim[1] = M (stride N)."""

    def __init__(self, shape, dtype, host_ptr=0, device_ptr=0, keepalive=None):
        # (every argument of every call that is given as a tensor or an array passes here: structures are filled in one
        # go, without an object per dimension)
        dtype = np.dtype(dtype)
        self.keepalive = keepalive
        self.shape, self.dtype, self.on_device = tuple([int(v) for v in shape]), dtype, bool(device_ptr)
        nd = len(self.shape)
        self.dims = (halide_dimension_t * max(nd, 1))()
        stride, numbers = 1, []
        for extent in reversed(self.shape):
            numbers += (0, extent, stride, 0)
            stride *= extent
        self.elements = stride
        try:
            struct.pack_into("=%di" % len(numbers), self.dims, 0, *numbers)
        except struct.error:                    # beyond 31 bits: the fields hold the low 32 of them
            for i in range(nd):
                self.dims[i] = halide_dimension_t(*numbers[4 * i:4 * i + 4])
        self.raw = halide_buffer_t(device_ptr, None, host_ptr, 0, (_TYPE_CODES[dtype.kind], dtype.itemsize * 8, 1), nd,
                                   _DIMENSIONS_OF.from_buffer(ctypes.c_void_p(ctypes.addressof(self.dims))))

    @staticmethod
    def from_numpy(a):
        if not a.flags["C_CONTIGUOUS"]:
            raise ValueError("Tiramisu buffers are dense row-major: pass a C-contiguous array")
        return Buffer(a.shape, a.dtype, host_ptr=a.ctypes.data, keepalive=a)

    @staticmethod
    def from_device(ptr, shape, dtype, keepalive=None):
        """A buffer that already lives in GPU memory (an argument tagged tag_gpu_global())."""
        return Buffer(shape, dtype, host_ptr=0, device_ptr=int(ptr), keepalive=keepalive)

    @staticmethod
    def from_tensor(t):
        """A ``torch.Tensor`` as an argument, without a copy: a tensor on the GPU describes a buffer tagged
        tag_gpu_global() (its storage is the device pointer), a CPU tensor a host buffer.  bfloat16 tensors
        are the 16-bit storage of p_bfloat16 buffers.  The tensor stays referenced while the buffer lives."""
        if not t.is_contiguous():
            raise ValueError("Tiramisu buffers are dense row-major: pass a contiguous tensor")
        dtype = _tensor_type(t.dtype)
        if t.is_cuda:
            return Buffer(t.shape, dtype, device_ptr=t.data_ptr(), keepalive=t)
        return Buffer(t.shape, dtype, host_ptr=t.data_ptr(), keepalive=t)

    def pointer(self):
        return ctypes.byref(self.raw)


_wrappers = None


def wrappers():
    """The runtime C ABI (include/tiramisu_hip_wrappers.h), loaded with global symbol visibility
    so that program libraries resolve against it."""
    global _wrappers
    if _wrappers is None:
        path = _build.wrappers_library()
        if not os.path.exists(path):
            raise RuntimeError("%s is missing: run __graft_entry__.build() first" % path)
        lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        lib.tiramisu_hip_malloc.restype = ctypes.c_void_p
        lib.tiramisu_hip_malloc.argtypes = [ctypes.c_uint64]
        lib.tiramisu_hip_free.argtypes = [ctypes.c_void_p]
        for fn in (lib.tiramisu_hip_memcpy_to_device, lib.tiramisu_hip_memcpy_to_host,
                   lib.tiramisu_hip_memcpy_device_to_device):
            fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64]
        lib.tiramisu_hip_stream_synchronize.argtypes = [ctypes.c_int32]
        lib.tiramisu_hip_set_stream.argtypes = [ctypes.c_void_p]
        lib.tiramisu_hip_get_stream.restype = ctypes.c_void_p
        lib.tiramisu_hip_stream_create.restype = ctypes.c_void_p
        lib.tiramisu_hip_stream_destroy.argtypes = [ctypes.c_void_p]
        lib.tiramisu_hip_call.argtypes = [ctypes.c_void_p, ctypes.c_int32] + [ctypes.c_void_p] * 3
        lib.tiramisu_hip_sgemm_workspace.restype = ctypes.c_void_p
        lib.tiramisu_hip_kept_scratch.restype = ctypes.c_void_p
        lib.tiramisu_hip_kept_scratch.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.POINTER(ctypes.c_int32)]
        lib.tiramisu_hip_release_cached_memory.restype = ctypes.c_uint64
        lib.tiramisu_hip_cached_memory_bytes.restype = ctypes.c_uint64
        lib.tiramisu_hip_event_create.restype = ctypes.c_void_p
        lib.tiramisu_hip_event_record.argtypes = [ctypes.c_void_p]
        lib.tiramisu_hip_event_elapsed_ms.restype = ctypes.c_float
        lib.tiramisu_hip_event_elapsed_ms.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        lib.tiramisu_hip_event_destroy.argtypes = [ctypes.c_void_p]
        lib.tiramisu_hip_profile_name.restype = ctypes.c_char_p
        lib.tiramisu_hip_profile_name.argtypes = [ctypes.c_int]
        lib.tiramisu_hip_profile_ms.restype = ctypes.c_float
        lib.tiramisu_hip_profile_ms.argtypes = [ctypes.c_int]
        u64 = ctypes.c_uint64
        lib.tiramisu_hip_sgemm.argtypes = [ctypes.c_void_p] * 3 + [u64] * 3 + [ctypes.c_float] * 2 + \
            [u64] * 6 + [ctypes.c_bool] * 2
        lib.tiramisu_hip_sgemm_static_scratch.argtypes = lib.tiramisu_hip_sgemm.argtypes
        lib.tiramisu_hip_dgemm.argtypes = [ctypes.c_void_p] * 3 + [u64] * 3 + [ctypes.c_double] * 2 + \
            [u64] * 6 + [ctypes.c_bool] * 2
        _wrappers = lib
    return _wrappers


_C_TYPES = {"float": "float32", "double": "float64", "int8_t": "int8", "int16_t": "int16", "int32_t": "int32", "int64_t": "int64",
            "uint8_t": "uint8", "uint16_t": "uint16", "uint32_t": "uint32", "uint64_t": "uint64", "bool": "bool",
            "tiramisu_bf16_t": "uint16"}


def manifest_of(library_path, function_name):
    """The description the HIP back-end writes next to each object (``<object>.json``: arguments
    with type, shape and memory space, kernels emitted) for the object that ``lib<stem>.so`` was
    linked from (``<stem>.o`` or ``generated_fct_<stem>.o`` in the same directory), or None."""
    import json
    directory, base = os.path.split(os.path.abspath(library_path))
    stem = base[3:-3] if base.startswith("lib") and base.endswith(".so") else base
    for name in (stem + ".o.json", "generated_fct_" + stem + ".o.json"):
        path = os.path.join(directory, name)
        if os.path.exists(path):
            try:
                m = json.load(open(path))
            except ValueError:
                return None
            return m if m.get("function") == function_name else None
    return None


class Program:
    """One compiled Tiramisu function: ``Program(path, "test_167")(A, B, C)`` with numpy arrays
    and/or ``Buffer`` objects as arguments.  When the back-end's description of the function is
    found next to the library, arguments are checked against it before the call (count, element
    type, constant extents, host or device memory): a wrong buffer would otherwise be a
    out-of-bounds access on the GPU."""

    expected = None          # _expected_arguments(), from the first check on

    def __init__(self, library_path, function_name, needs_gpu_runtime=True):
        if not os.path.exists(library_path):
            raise RuntimeError("%s is missing: run __graft_entry__.build() first" % library_path)
        if needs_gpu_runtime:
            wrappers()
        self.lib = ctypes.CDLL(library_path)
        self.fn = getattr(self.lib, function_name)
        self.fn.restype = ctypes.c_int
        self.name = function_name
        self.manifest = manifest_of(library_path, function_name) if needs_gpu_runtime else None
        self.loaded = self.fn

    def _expected_arguments(self):
        """What check() compares: (description, element type, on the device, number of elements) of every argument,
        None where anything will do."""
        out = []
        for e in self.manifest["arguments"]:
            # a host input may be declared larger than what the program reads of it (the reference's
            # sgemm generators declare their two scalars over the row range); anything the GPU
            # touches, and every output, must have the declared number of elements
            strict = e["memory"] == "device" or e["kind"] != "input"
            constant = strict and all(isinstance(v, int) for v in e["shape"])
            out.append((e, np.dtype(_C_TYPES[e["type"]]) if e["type"] in _C_TYPES else None, e["memory"] == "device",
                        math.prod(e["shape"]) if constant else None))
        return out

    @functools.cached_property
    def of_tensors(self):
        """For calls whose arguments are all GPU tensors: the function, its address, the declared (element type, shape) of every argument,
        and what tiramisu_hip_call takes.  None where an argument lives on the host or has no literal shape.  Made at the first call with a
        tensor: programs that only see buffers need none of it (loading one took 56 us with it, 43 without)."""
        fn, arguments, description = self.loaded, [], []
        if self.manifest is None:
            return None
        for e in self.manifest["arguments"]:
            shape = e["shape"]
            if e["memory"] != "device" or e["type"] not in _C_TYPES or len(shape) > 8 or not all(isinstance(v, int) and 0 < v < 1 << 31 for v in shape):
                return None
            dtype = np.dtype(_C_TYPES[e["type"]])
            arguments.append((dtype, tuple(shape)))
            description += [_TYPE_CODES[dtype.kind], dtype.itemsize * 8, len(shape)] + shape
        if not 1 <= len(arguments) <= 8:
            return None
        return (fn, ctypes.cast(fn, ctypes.c_void_p).value, tuple(arguments), struct.Struct("=%dQ" % len(arguments)).pack,
                struct.pack("=%di" % len(description), *description))

    def _call_of_tensors(self, args):
        """A call whose arguments are all dense GPU tensors of the declared types and shapes, through one entry of the runtime (a structure
        per argument made here, and four entries: a convolution 3 to 64 channels, of which 12 us are the kernel, 37.3 us a call; so 24.9).
        None if they are not: the general way looks closer, and says what does not fit."""
        fn, address, arguments, pack_pointers, description = self.of_tensors
        torch = sys.modules.get("torch")
        if torch is None or self.fn is not fn or len(args) != len(arguments):
            return None
        kinds, pointers = (torch.Tensor, torch.nn.Parameter), []
        for a, (dtype, shape) in zip(args, arguments):
            if type(a) not in kinds or _tensor_type(a.dtype) is not dtype or a.shape != shape or not a.is_cuda or not a.is_contiguous():
                return None
            pointers.append(a.data_ptr())
        if 0 in pointers:
            return None
        raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
        stream = raw_stream(args[0].get_device()) if raw_stream else torch.cuda.current_stream(args[0].device).cuda_stream
        return wrappers().tiramisu_hip_call(address, len(pointers), pack_pointers(*pointers), description, stream)

    def check(self, bufs):
        if self.expected is None:
            self.expected = self._expected_arguments()
        if len(bufs) != len(self.expected):
            raise ValueError("%s takes %d buffers, %d given" % (self.name, len(self.expected), len(bufs)))
        for b, (e, dtype, on_device, elements) in zip(bufs, self.expected):
            if dtype is not None and dtype != b.dtype:
                raise ValueError("%s: buffer %s holds %s, %s given" % (self.name, e["name"], e["type"], b.dtype))
            if on_device != b.on_device:
                raise ValueError("%s: buffer %s lives in %s memory" % (self.name, e["name"], e["memory"]))
            if elements is not None and b.elements != elements:
                raise ValueError("%s: buffer %s has shape %s, %s given" % (self.name, e["name"], e["shape"], list(b.shape)))

    def __call__(self, *args):
        """Arguments: ``Buffer`` objects, numpy arrays (host buffers) or torch tensors (host or GPU buffers by where
        they live).  With a GPU tensor among them the function's kernels run on torch's current stream of that
        tensor's device, in order with the torch work around the call (the runtime's stream of the calling thread is
        put back afterwards); when that is torch's default stream they run on the runtime's stream of the calling
        thread, and the call waits for torch's default stream first and for its own kernels afterwards."""
        bufs, torch_stream = [], None
        for a in args:
            if isinstance(a, Buffer):
                bufs.append(a)
            elif isinstance(a, np.ndarray):
                bufs.append(Buffer.from_numpy(a))
            elif type(a).__module__.split(".")[0] == "torch":
                if not bufs and self.of_tensors is not None:
                    rc = self._call_of_tensors(args)
                    if rc is not None:
                        if rc != 0:
                            raise RuntimeError("Tiramisu function returned %d" % rc)
                        return rc
                bufs.append(Buffer.from_tensor(a))
                if a.is_cuda and torch_stream is None:
                    import torch
                    torch_stream = torch.cuda.current_stream(a.device).cuda_stream
            else:
                bufs.append(Buffer.from_numpy(a))
        if self.manifest is not None:
            self.check(bufs)
        if torch_stream is None:
            rc = self.fn(*[b.pointer() for b in bufs])
        elif torch_stream == 0:
            # torch's default stream is the device's null stream, and its handle, 0, means the calling thread's own default
            # stream to tiramisu_hip_set_stream.  The kernels stay on the thread's stream, so that calls from several threads
            # overlap (two threads of a 1.33 ms pass each 2.0 to 2.2 ms a round; on the null stream, one after the other, 2.7),
            # ordered by a wait on both sides.  The runtime waits: torch's synchronize() costs 3 us more.
            w = wrappers()
            w.tiramisu_hip_null_stream_synchronize()
            rc = self.fn(*[b.pointer() for b in bufs])
            w.tiramisu_hip_stream_synchronize(0)
        else:
            w = wrappers()
            before = w.tiramisu_hip_get_stream()
            w.tiramisu_hip_set_stream(torch_stream)
            try:
                rc = self.fn(*[b.pointer() for b in bufs])
            finally:
                w.tiramisu_hip_set_stream(before)
        if rc != 0:
            raise RuntimeError("Tiramisu function returned %d" % rc)
        return rc


def load(directory, name, function_name=None):
    return Program(_build.program_library(directory, name), function_name or name)


def profile(fn):
    """Run ``fn()`` with per-launch timing on; returns [(kernel name, milliseconds), ...]."""
    w = wrappers()
    w.tiramisu_hip_profile_start()
    fn()
    n = w.tiramisu_hip_profile_stop()
    return [(w.tiramisu_hip_profile_name(i).decode(), float(w.tiramisu_hip_profile_ms(i))) for i in range(n)]


class DeviceTimer:
    """HIP-event timing on the stream that generated code launches on."""

    def __init__(self):
        self.w = wrappers()
        self.start = self.w.tiramisu_hip_event_create()
        self.stop = self.w.tiramisu_hip_event_create()

    def __enter__(self):
        self.w.tiramisu_hip_event_record(self.start)
        return self

    def __exit__(self, *exc):
        self.w.tiramisu_hip_event_record(self.stop)
        self.ms = self.w.tiramisu_hip_event_elapsed_ms(self.start, self.stop)
        return False
