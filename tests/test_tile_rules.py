"""The sweeps' tile grids and the choice of their shape (sweep_grid, fewest_blocks in
csrc/xf_context.h) over all sizes, on the host: every cell and column lies in exactly one
tile, no tile exceeds its lanes or is empty, directions without cells give no tiles, and
an ensemble's shape does not depend on the order of its cases."""
import shutil
import subprocess

import pytest

from xfluids_amd import build

SOURCE = r"""
#include "%s/csrc/xf_context.h"
#include <cstdio>
using namespace xf;
static Geom geom(int x, int y, int z)
{
    Geom g{};
    g.X_inner = x, g.Y_inner = y, g.Z_inner = z;
    return g;
}
static int failed(const char *what, int x, int y, int z, int dir, int shape, long long launch)
{
    std::printf("%%s: %%d x %%d x %%d direction %%d shape %%d launch %%lld\n", what, x, y, z, dir, shape, launch);
    return 1;
}
// the tiles of n cells by span cover each once: the last one is not empty
static bool covers(int n, unsigned tiles, unsigned span, int most)
{
    return span >= 1 && (int)span <= most && (long long)tiles * span >= n && (long long)(tiles - 1) * span < n;
}
int main()
{
    int bad = 0;
    for (int n = 1; n <= 700; n++)
        for (int m : {1, 2, 7, 8, 16, 31, 32, 33, 250, 700})
            for (int dir = 0; dir < 3; dir++)
                for (int s = 0; s < (dir == 0 ? 2 : 3); s++) {
                    const int x = dir == 0 ? n : m, y = dir == 1 ? n : 5, z = dir == 2 ? n : 3;
                    const Geom g = geom(x, y, z);
                    const int TS = tile_faces(dir, s), TW = 256 / TS;
                    unsigned r[5];
                    for (long long launch : {0LL, 511LL, 512LL, 100000LL}) {
                        sweep_grid(g, dir, s, launch, r);
                        const unsigned along = dir == 0 ? r[0] : r[1], across = dir == 0 ? r[1] : r[0];
                        if (!covers(n, along, r[3], TS - 1)) bad += failed("cells", x, y, z, dir, s, launch);
                        if (!covers(dir == 0 ? y * z : x, across, dir == 0 ? TW : r[4], TW))
                            bad += failed("columns", x, y, z, dir, s, launch);
                        if (r[2] != (unsigned)(dir == 0 ? 1 : (dir == 1 ? z : y))) bad += failed("third", x, y, z, dir, s, launch);
                        if ((long long)r[0] * r[1] * r[2] != tile_blocks(g, dir, s)) bad += failed("blocks", x, y, z, dir, s, launch);
                    }
                }
    // grids without cells in a direction, which xf_create takes: no tiles
    for (int dir = 0; dir < 3; dir++)
        for (int s = 0; s < (dir == 0 ? 2 : 3); s++)
            for (int n : {0, -2})
                for (int axis = 0; axis < 3; axis++) {
                    const int x = axis == 0 ? n : 16, y = axis == 1 ? n : 16, z = axis == 2 ? n : 16;
                    unsigned r[5];
                    for (long long launch : {0LL, 100000LL}) {
                        sweep_grid(geom(x, y, z), dir, s, launch, r);
                        std::printf("empty %%u\n", r[0] + r[1] + r[2] + r[3] + r[4]);
                    }
                }
    // the order of an ensemble's cases
    const Geom a = geom(64, 7, 1), b = geom(256, 256, 1);
    for (int dir = 0; dir < 2; dir++) {
        auto of = [&](const Geom *g, int n) {
            return fewest_blocks(dir, [&](int s) {
                long long sum = 0;
                for (int k = 0; k < n; k++) sum += tile_blocks(g[k], dir, s);
                return sum;
            });
        };
        const Geom ab[3] = {a, b, b}, ba[3] = {b, b, a};
        if (of(ab, 3) != of(ba, 3) || (dir == 1 && (of(&a, 1) != 2 || of(ab, 3) != 0)))
            bad += failed("order", 0, 0, 0, dir, 0, 0);
    }
    return bad != 0;
}
"""


@pytest.mark.skipif(not shutil.which(build.HIPCC), reason="no hipcc")
def test_tile_rules(tmp_path):
    src, exe = tmp_path / "rules.hip", tmp_path / "rules"
    src.write_text(SOURCE % build.PKG)
    subprocess.run([build.HIPCC, "--offload-host-only", "-x", "hip", "-O1", "-std=c++17", "-I", build.ROOT + "/include",
                    str(src), "-o", str(exe)], check=True, capture_output=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-500:]
