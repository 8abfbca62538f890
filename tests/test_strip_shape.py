"""Which blocks a grid takes on the strip kernel (csrc/strip_shape.h), compiled
here with the host compiler: every grid's workgroup fits (threads, LDS, whole
blocks where the shape needs them), the grids that measured one shape well
ahead of the others take it or one close to it, and the grids that the GPU
tests name reach every form of the kernel (shape, in two phases or one)."""
import os
import shutil
import subprocess

import pytest

import strip_grids

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "latticemodels.jl_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include "strip_shape.h"
using namespace lmh;
int main() {
    int lx, ly;
    while (std::scanf("%d %d", &lx, &ly) == 2) {
        StripGeom g;
        const bool ok = strip_shape(lx, ly, &g);
        StripGeom b;
        const bool okb = strip_batch_shape(lx, ly, &b);
        std::printf("%d %d %d %d %d %d %d %d %d\n", lx, ly, ok ? g.bx : 0, ok ? g.s : 0, g.threads, g.cols, g.nthr,
                    okb ? b.bx : 0, okb ? b.s : 0);
    }
    // every grid: what the kernel and its launcher take for granted
    long bad = 0, grids = 0, strips = 0;
    for (int x = 2; x <= 2560; ++x)
        for (int y = 4; x * y <= 10240; ++y)
            for (int batch = 0; batch < 2; ++batch) {
            StripGeom g;
            ++grids;
            if (!(batch ? strip_batch_shape(x, y, &g) : strip_shape(x, y, &g))) continue;
            ++strips;
            if (batch) {
                const int c = strip_batch_cols(g);
                if (c < 1 || c * g.nthr > 512 || 16L * g.region * c > 163840) ++bad;
            }
            const int nbx = (x + g.bx - 1) / g.bx;
            const bool whole = x % g.bx == 0 && y % g.s == 0;
            if (g.lx != x || g.ly != y || g.bx > x || g.s > y || g.q != (y + g.s - 1) / g.s || g.nt != x * g.q ||
                g.nthr != nbx * g.q || g.threads % 64 || g.threads < 64 || g.threads > 512 || g.cols < 1 ||
                g.cols * g.nthr > g.threads || g.lyp < g.bx * y || g.lyp % 2 == 0 || g.region < nbx * g.lyp + 1 ||
                16L * g.region * g.cols > 163840 || (g.bx > 2 && !whole))
                ++bad;
        }
    std::printf("all %ld %ld %ld\n", grids, strips, bad);
}
"""


def _harness(tmp_path, grids):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "h.cpp", tmp_path / "h"
    src.write_text(HARNESS)
    subprocess.check_call([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)])
    text = "\n".join("%d %d" % g for g in grids)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
    return [tuple(int(v) for v in line.split()) for line in out[: len(grids)]], out[len(grids)]


# us per step by shape where the shapes differ most (the rest within 10 % of the best)
MEASURED = {
    (37, 23): {(2, 4): 33.6, (2, 6): 40.2, (2, 8): 40.4, (2, 10): 44.8, (1, 20): 62.7},
    (61, 42): {(2, 6): 186, (2, 10): 268},
    (100, 100): {(2, 10): 2365, (1, 20): 2672},
    (2, 1000): {(2, 5): 104, (2, 10): 108, (1, 20): 108, (2, 6): 124, (2, 4): 125, (2, 8): 189},
    (2, 2000): {(2, 5): 407, (1, 20): 414, (2, 10): 420, (2, 6): 486, (2, 4): 523, (2, 8): 776},
    (3, 2000): {(2, 10): 1158, (1, 20): 1252, (2, 8): 1830},
    (4, 2000): {(2, 10): 1664, (1, 20): 1724, (4, 4): 1857, (2, 8): 2547},
    (5, 1000): {(1, 20): 658, (2, 6): 730, (2, 10): 916, (2, 8): 1082},
    (6, 1200): {(2, 10): 1514, (1, 20): 1615, (2, 8): 1917},
    (7, 700): {(1, 20): 650, (2, 6): 702, (2, 8): 828, (2, 10): 881},
    (11, 85): {(2, 5): 36.4, (2, 6): 41.1, (2, 10): 43.9, (1, 20): 45.0, (2, 4): 50.0, (2, 8): 50.4},
    (300, 5): {(2, 5): 105, (2, 4): 187},
    (340, 5): {(2, 5): 158, (2, 4): 218},
}


# the same in uniform batches (us per step of all members)
BATCHES = {
    (35, 35): {(2, 5): 979, (2, 6): 1066, (2, 4): 1071, (1, 20): 1116, (2, 8): 1145, (2, 10): 1162},
    (64, 40): {(4, 4): 1777, (2, 5): 1854, (2, 8): 1925, (2, 6): 1990, (2, 10): 2144, (1, 20): 2187, (2, 4): 2631},
    (25, 100): {(1, 20): 1920, (2, 8): 2072, (2, 6): 2095, (2, 10): 2265, (2, 4): 2833, (2, 5): 3165},
    (5, 400): {(1, 20): 1566, (2, 10): 1801, (2, 5): 1835, (2, 6): 2035, (2, 8): 2495, (2, 4): 2969},
    (2, 300): {(2, 6): 468, (2, 5): 471, (1, 20): 477, (2, 10): 490, (2, 4): 634, (2, 8): 858},
    (2, 1000): {(2, 10): 1395, (1, 20): 1400, (2, 6): 1423, (2, 5): 1543, (2, 4): 1860, (2, 8): 2756},
    (3, 340): {(1, 20): 869, (2, 10): 983, (2, 6): 986, (2, 5): 1124, (2, 4): 1181, (2, 8): 1397},
}


def test_every_grid_fits_and_measured_grids_take_a_fast_shape(tmp_path):
    rows, everything = _harness(tmp_path, list(MEASURED))
    assert everything.split()[3] == "0" and int(everything.split()[2]) > 30000
    for lx, ly, bx, s, *_ in rows:
        times = MEASURED[(lx, ly)]
        assert times[(bx, s)] <= 1.1 * min(times.values()), (lx, ly, bx, s)
    rows, _ = _harness(tmp_path, list(BATCHES))
    for lx, ly, *_, bx, s in rows:
        times = BATCHES[(lx, ly)]
        assert times[(bx, s)] <= 1.1 * min(times.values()), (lx, ly, bx, s)


def test_grids_of_the_gpu_tests_reach_every_form(tmp_path):
    rows, _ = _harness(tmp_path, [g[:2] for g in strip_grids.FORMS])
    reached = set()
    for (lx, ly, bx, s, *_), (_, _, shape, phases) in zip(rows, strip_grids.FORMS):
        assert (bx, s) == shape and (bx > 2 or ly % s == 0) == phases
        reached.add((shape, phases))
    shapes = [(1, 20), (2, 10), (2, 8), (2, 6), (2, 5), (2, 4)]
    assert reached == {(sh, p) for sh in shapes for p in (True, False)} | {((4, 4), True)}


def test_a_grid_too_wide_for_its_blocks_has_no_strips(tmp_path):
    rows, _ = _harness(tmp_path, [(600, 5), (300, 33), (2, 3000)])
    assert [r[2] for r in rows] == [0, 0, 2]
