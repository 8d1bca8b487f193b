"""fp64 products whose 96 x 96 tiles share their slices of 32 k between two groups of wavefronts (kernels/gemm_mfma_f64.hip.h), at one row or
column behind a tile and with 26, 1 and no k in the last slice, and the 96 x 96 tiles that do not; exact for integers."""
import os
import re
import subprocess

import numpy as np
import pytest

from test_library_gemm import surrounded_by_nan
from tiramisu_amd import build

SIZES = [(1500, 1430, 250, 7), (1535, 1441, 289, 7), (1440, 1536, 320, 7), (2400, 2232, 318, 1)]
# 32 x 32 tiles (3) are faster where the k are few, 96 x 96 with shared slices where they are many
LINE = [(1664, 1337, 140, 3), (1943, 1135, 170, 3), (1184, 1736, 384, 3), (1184, 1698, 672, 7), (1029, 1947, 580, 7), (1248, 1663, 1109, 7), (904, 1646, 991, 3)]


def test_rule(tmp_path):
    """The rule as the header states it: which tile each size takes (7: 96 x 96 with shared slices, 1: without)."""
    text = open(os.path.join(build.CSRC, "kernels", "gemm_mfma_f64.hip.h")).read()
    rule = re.search(r"enum tile \{.*?\};", text, re.S).group(0) + re.search(r"inline tile tile_for\(.*?\n\}", text, re.S).group(0)
    (tmp_path / "rule.cpp").write_text('#include <cstdio>\n#include "%s"\n%s\nint main() {\n%s}\n' % (
        os.path.join(build.CSRC, "kernels", "target_gfx950.h"), rule, "".join('    printf("%%d ", tile_for(%d, %d, %d));\n' % s[:3] for s in SIZES + LINE)))
    subprocess.run(["g++", "-std=c++17", "-o", str(tmp_path / "rule"), str(tmp_path / "rule.cpp")], check=True)
    assert [int(v) for v in subprocess.run([str(tmp_path / "rule")], stdout=subprocess.PIPE, text=True).stdout.split()] == [s[3] for s in SIZES + LINE]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile", SIZES)
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("pad", [0, 3])
def test_inside_larger_allocations(M, N, K, tile, tA, tB, pad):
    surrounded_by_nan(M, N, K, tA, tB, pad, np.float64)
