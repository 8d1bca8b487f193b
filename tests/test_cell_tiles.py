"""Tiles of recurrent cells on at most 64 rows: 32x32 shared by groups of wavefronts where the launch leaves the chip idle, at its edges and
on both sides of the rule, against the oracle (tolerance of test_lstm.py: fp32 sums in another order)."""
import json
import os

import numpy as np
import pytest

from oracle import reference_loops as ref
from test_lstm import RTOL, make_inputs, name_of
from tiramisu_amd import runtime

CASES = [((2, 33, 40, 5), "tile 32x32x64, guarded", True), ((3, 5, 24, 4), "tile 32x32x64, guarded", True), ((2, 9, 37, 3), "tile 32x32x64, guarded", False),
         ((1, 64, 384, 3), "tile 32x32x128, whole", True), ((2, 64, 512, 4), "tile 32x32x64, whole", True), ((4, 64, 512, 5), "tile 64x32x64, whole", True)]


@pytest.mark.parametrize("s,what,fused", CASES)
def test_tile(s, what, fused, programs_dir):
    kernels = json.load(open(os.path.join(programs_dir, "build", name_of(s) + ".o.json")))["kernels"]
    cells = [k["how"] for k in kernels if "tile " in k["how"]]
    assert cells and all(what in h for h in cells)
    assert any("point-wise statement" in h for h in cells) == fused


@pytest.mark.gpu
@pytest.mark.parametrize("s", [c[0] for c in CASES])
def test_gpu(s, programs_dir):
    from gpu_util import DeviceArray
    w, b, x = make_inputs(s, sum(s))
    d = [DeviceArray(a) for a in (w, b, x, np.full((s[3], s[1], s[2]), np.nan, np.float32))]
    runtime.load(programs_dir, name_of(s))(*[q.buffer() for q in d])
    y, expected = d[3].download(), ref.lstm(w, b, x)
    assert np.max(np.abs(y - expected)) <= RTOL * np.max(np.abs(expected))


GROUPS = [((64, 32, 16, 96), "tile 64x64x32"), ((64, 128, 4, 96), "tile 32x32x64")]


@pytest.mark.parametrize("s,tile", GROUPS)
def test_column_groups_stay_in_one_launch(s, tile, programs_dir):
    """A product and the nest that adds its column groups are one kernel, also where tiles of 32 columns hold too few units of them."""
    kernels = json.load(open(os.path.join(programs_dir, "build", "column_groups_%dx%dx%dx%d.o.json" % s)))["kernels"]
    assert len(kernels) == 1 and tile in kernels[0]["how"] and "(%d column group(s) per unit, 1 temporaries kept in registers)" % s[2] in kernels[0]["how"]


@pytest.mark.gpu
@pytest.mark.parametrize("s", [g[0] for g in GROUPS])
def test_gpu_column_groups(s, programs_dir):
    from gpu_util import DeviceArray
    M, H, G, K = s
    rng = np.random.RandomState(G)
    a, w = rng.randint(-4, 5, (M, K)).astype(np.float32), rng.randint(-4, 5, (K, G * H)).astype(np.float32)
    d = [DeviceArray(v) for v in (a, w, np.full((M, H), np.nan, np.float32))]
    runtime.load(programs_dir, "column_groups_%dx%dx%dx%d" % s)(*[q.buffer() for q in d])
    assert np.array_equal(d[2].download(), (a @ w).reshape(M, G, H).sum(1))
