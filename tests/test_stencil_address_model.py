"""The stencil kernel's loads and stores, enumerated on the host.

tests/host_models/stencil_address_model.cpp compiles kernels/stencil2d_regs.hip.h itself as plain C++ (its
host-model form: every access to global memory is recorded instead of performed) and runs every workgroup and
thread of every launch that the emitter's plan (csrc/stencil_plan.h) makes for plane sizes 5 ... 300 (every
residue mod 4, square and not), 1 ... 13 steps per launch and the four kernel modes, as far as they take the instance of
the kernel that was compiled (the program prints how many do): loads inside their buffer
and aligned, every cell a launch owes written exactly once and nothing else, whole time loops ending with the
right steps in the right planes.  The second test breaks the kernel's indexing in a copy and expects the model
to say so: a model that cannot fail pins nothing.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MODEL = os.path.join(ROOT, "tests", "host_models", "stencil_address_model.cpp")


def build_model(source, out, *defines):
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wno-unknown-pragmas", *defines, "-o", out, source], check=True)


def test_every_load_and_store_of_the_stencil_kernel_is_in_bounds_and_owed(tmp_path):
    exe = str(tmp_path / "model")
    build_model(MODEL, exe)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    print(r.stdout[-2000:])
    assert r.returncode == 0, r.stdout[-2000:]
    assert " 0 failure(s)" in r.stdout


# rows per thread of a strip and of a boundary slice: what the plan gives to planes that leave compute units idle, and (4, 2), a
# slice shorter than the strip at few rows
STRIPS = [(2, 2), (3, 3), (4, 2), (4, 4), (5, 2), (5, 5), (6, 3), (6, 6), (7, 3), (7, 7), (8, 4), (9, 4), (10, 5)]


def test_the_strips_are_those_that_the_plan_emits(tmp_path):
    source, exe = tmp_path / "strips.cpp", str(tmp_path / "strips")
    source.write_text('''#include "%s"
#include <cstdio>
#include <set>
int main() {
    std::set<std::pair<int, int>> strips;
    for (int ny = 20; ny <= 8192; ny += ny < 700 ? 3 : ny < 3000 ? 17 : 61)
        for (int nx : {ny, 20, 300, 777, 2049, 8192})
            for (int steps = 1; steps <= 32; steps++)
                for (const tstencil::chunk &c : tstencil::plan_time_loop(1, steps, tstencil::step_cap(12, 1, 88), false, steps >= 3)) {
                    const int rows = tstencil::plan_rows(ny, nx, 1, ny - 2, 1, nx - 2, 1, c.steps, 8, 11);
                    strips.insert({rows, tstencil::plan_launch(ny, nx, 1, ny - 2, 1, nx - 2, 1, c.steps, 8, rows).rows_edge});
                }
    for (auto &s : strips) std::printf("%%d %%d\\n", s.first, s.second);
}
''' % os.path.join(ROOT, "tiramisu_amd", "csrc", "stencil_plan.h"))
    build_model(str(source), exe)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True).stdout
    emitted = {tuple(int(v) for v in line.split()) for line in out.splitlines()}
    assert emitted == set(STRIPS) - {(4, 2)} | {(11, 5)}


@pytest.mark.parametrize("rows,rows_edge", STRIPS)
def test_fewer_rows_per_thread(tmp_path, rows, rows_edge):
    """The strips that the plan gives to small planes: planes of one tile to several, with and without interior tiles, down to
    tiles of the fewest rows; of the numbers of steps those whose slices have the given rows (the model says how many
    launches that were, and fails at none)."""
    exe = str(tmp_path / "model")
    build_model(MODEL, exe, "-DMODEL_ROWS=%d" % rows, "-DMODEL_ROWS_EDGE=%d" % rows_edge)
    for lo, hi in ((5, 40), (530, 532)):
        r = subprocess.run([exe, str(lo), str(hi), "12"], stdout=subprocess.PIPE, text=True)
        print(r.stdout[-300:])
        assert r.returncode == 0 and " 0 failure(s)" in r.stdout, r.stdout[-2000:]


def test_the_model_fails_where_it_runs_no_launch(tmp_path):
    exe = str(tmp_path / "model")
    build_model(MODEL, exe, "-DMODEL_ROWS=2", "-DMODEL_ROWS_EDGE=1")         # (a slice of one row: the plan makes none)
    r = subprocess.run([exe, "5", "10", "3"], stdout=subprocess.PIPE, text=True)
    assert r.returncode != 0 and "FAIL no fused launch" in r.stdout


def test_the_values_of_quads_at_the_edges_of_a_plane(tmp_path):
    """Rows of every length, so that every shift of a quad that hangs over a row's end occurs; a mistake in one of them is reported."""
    exe, source = str(tmp_path / "quads"), os.path.join(ROOT, "tests", "host_models", "stencil_quad_model.cpp")
    build_model(source, exe)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0 and " 0 wrong value(s), 0 load(s) outside" in r.stdout, r.stdout[-2000:]
    header = os.path.join(ROOT, "tiramisu_amd", "csrc", "kernels", "stencil2d_regs.hip.h")
    text = open(header).read()
    for old, new in (("behind == 1 ? one", "behind == 1 ? two"), ("behind == 2 ? two : three", "behind == 2 ? three : two"), ("gx - at;", "gx - at - 1;")):
        assert text.count(old) == 1, old
        (tmp_path / "stencil2d_regs.hip.h").write_text(text.replace(old, new))
        shutil.copy(os.path.join(os.path.dirname(header), "target_gfx950.h"), tmp_path)
        broken = tmp_path / "broken.cpp"
        broken.write_text(open(source).read().replace("../../tiramisu_amd/csrc/kernels/", ""))
        build_model(str(broken), exe)
        r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
        assert r.returncode != 0 and "FAIL" in r.stdout, "accepted: " + new


def test_the_model_reports_broken_indexing(tmp_path):
    """Three one-token mistakes in a copy of the kernel: a tile one row too tall, a strip one lane too wide, a
    region shifted by one quad.  Each must be reported."""
    tree = tmp_path / "copy"
    (tree / "tests" / "host_models").mkdir(parents=True)
    (tree / "tiramisu_amd" / "csrc" / "kernels").mkdir(parents=True)
    shutil.copy(MODEL, tree / "tests" / "host_models")
    shutil.copy(os.path.join(ROOT, "tiramisu_amd", "csrc", "stencil_plan.h"), tree / "tiramisu_amd" / "csrc")
    kernels = os.path.join(ROOT, "tiramisu_amd", "csrc", "kernels")
    for h in ("stencil2d_regs.hip.h", "target_gfx950.h"):
        shutil.copy(os.path.join(kernels, h), tree / "tiramisu_amd" / "csrc" / "kernels")
    original = open(os.path.join(kernels, "stencil2d_regs.hip.h")).read()
    mistakes = [("gy >= row_end) continue;", "gy > row_end) continue;", ["5", "60", "5"]),
                ("4 * lane < ST_HX + ST_TW)", "4 * lane <= ST_HX + ST_TW)", ["290", "300", "3"]),
                ("const int gx = ox - ST_HX + 4 * lane;", "const int gx = ox - ST_HX + 4 * lane + 4;", ["5", "40", "3"])]
    for old, new, sweep in mistakes:
        assert original.count(old) == 1, old
        (tree / "tiramisu_amd" / "csrc" / "kernels" / "stencil2d_regs.hip.h").write_text(original.replace(old, new))
        exe = str(tmp_path / "broken")
        build_model(str(tree / "tests" / "host_models" / "stencil_address_model.cpp"), exe)
        r = subprocess.run([exe] + sweep, stdout=subprocess.PIPE, text=True)
        assert r.returncode != 0 and "FAIL" in r.stdout, "the model accepted: " + new
