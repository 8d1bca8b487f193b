"""Convolutions whose window is gathered (kernels/target_gfx950.h: gathered_tile_for): every tile, at its remainders and whole, against the
oracle; exact for integers, within the bound of sums of K fp32 products otherwise."""
import json
import os

import numpy as np
import pytest

from oracle import reference_loops as ref
from test_conv2d import make_inputs, name_of
from tiramisu_amd import runtime

CASES = [((2, 41, 33, 13), "tile 32x32x64, guarded"), ((1, 64, 32, 8), "tile 32x32x64, whole"), ((1, 44, 15, 96), "tile 32x64x64, guarded"),
         ((3, 15, 8, 91), "tile 32x128x16, guarded"), ((8, 40, 50, 92), "tile 64x64x32, guarded"), ((7, 11, 35, 67), "tile 64x128x16, guarded"),
         ((1, 64, 64, 16), "tile 32x32x64, whole"), ((4, 64, 64, 64), "tile 64x64x64, whole")]


@pytest.mark.parametrize("s,what", CASES)
def test_tile(s, what, programs_dir):
    how = json.load(open(os.path.join(programs_dir, "build", name_of(s) + ".o.json")))["kernels"][0]["how"]
    assert what in how and "gathered operand" in how


@pytest.mark.gpu
@pytest.mark.parametrize("integer", [True, False])
@pytest.mark.parametrize("s", [c[0] for c in CASES])
def test_gpu(s, integer, programs_dir):
    from gpu_util import DeviceArray
    xp, w, b = make_inputs(s, sum(s), integer=integer)
    d = [DeviceArray(a) for a in (xp, w, b, np.full((s[0], s[2], s[3], s[3]), np.nan, np.float32))]
    runtime.load(programs_dir, name_of(s))(*[q.buffer() for q in d])
    out, expected = d[3].download(), ref.conv2d_bias_relu(xp, w, b)
    if integer:
        assert np.array_equal(out, expected)
    else:        # |error| <= K roundings of half a unit of the sum of the magnitudes
        size = ref.conv2d_bias_relu(np.abs(xp), np.abs(w), np.abs(b))
        assert np.all(np.abs(out - expected) <= (9 * s[1] + 4) * 2.0 ** -24 * size)
