"""Host checks of the launch-shape rules (openems_amd/csrc/oe_tiles.h), built
with the host compiler: no device is needed, so grids of any size can be asked
about."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include "oe_tiles.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
    for (int q = 1; q + 2 < argc; q += 3) {
        oe::Grid g{atoi(argv[q]), atoi(argv[q + 1]), atoi(argv[q + 2]), 0};
        g.N = (size_t)g.nx * g.ny * g.nz;
        const oe::Tiles t = oe::auto_tiles(g, 0);
        printf("%d %d %d %d %d %d\\n", t.vec, t.bx, t.by, t.ci, oe::sweep_lanes(g, true), oe::sweep_lanes(g, false));
    }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("tiles")
    (d / "tiles.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "openems_amd", "csrc"), str(d / "tiles.cpp"), "-o",
                    str(d / "tiles")], check=True)

    def ask(*shapes):
        args = [str(v) for s in shapes for v in s]
        out = subprocess.run([str(d / "tiles"), *args], capture_output=True, text=True, check=True).stdout
        names = ("vec", "bx", "by", "ci", "sweep", "sweep_ragged")
        return [dict(zip(names, map(int, line.split()))) for line in out.splitlines()]

    return ask


def test_wide_planes_take_scalar_lanes(rules):
    """float4 lanes hold a cell's place in its plane, one row past either end
    included, in 32 bits: planes too wide for that take scalar lanes, in a
    single engine's launches and in a sweep's."""
    shapes = [(2, ny, nz) for ny, nz in ((32768, 32800), (32768, 32768), (32766, 32768), (32764, 32768), (4, 1 << 28), (2, 1 << 28),
                                         (1 << 28, 4), (100, 100), (60, 32))]
    for (_, ny, nz), r in zip(shapes, rules(*shapes)):
        fits = (ny + 2) * nz * 4 < 2 ** 32
        assert (r["vec"], r["sweep"]) == ((4, 4) if fits else (1, 1)), (ny, nz)
        assert r["sweep_ragged"] == 1


def _work_groups(shape, r):
    nx, ny, nz = shape
    lanes = -(-nz // r["vec"])
    return -(-lanes // r["bx"]) * -(-ny // r["by"]) * -(-nx // r["ci"])


def test_every_cell_has_a_lane_and_every_launch_fits(rules):
    """bx by at most 256 lanes, and no more lanes in a launch than 2^32 hold,
    on grids of any proportion up to 2^32 cells."""
    shapes = [(1 << 30, 1, 1), (1 << 25, 1, 1), (1 << 28, 2, 4), (1 << 29, 1, 5), (300_000_000, 3, 3), (40_000_000, 1, 64), (1, 1, 1),
              (1 << 20, 64, 64), (512, 512, 512), (1 << 26, 8, 4), (1 << 16, 1 << 8, 1 << 8), (3, 1 << 29, 2), (2, 2, 1 << 30)]
    for s, r in zip(shapes, rules(*shapes)):
        assert 1 <= r["bx"] and 1 <= r["by"] and r["bx"] * r["by"] <= 256 and 1 <= r["ci"] <= s[0], (s, r)
        assert _work_groups(s, r) * 256 < 2 ** 32, (s, r)


def test_nearly_empty_planes_are_marched_deep(rules):
    """Planes that fill less than half of their lanes: no more than a few
    thousand work-groups for each sixteenfold depth; full ones as before."""
    thin = [(100_000, 4, 4), (1_000_000, 1, 1), (20_000, 16, 16), (2000, 1, 2000), (100_000, 8, 8), (200_000, 2, 2)]
    for s, r in zip(thin, rules(*thin)):
        assert r["ci"] > 2 and _work_groups(s, r) <= 20_000, (s, r)
    full = [((100, 100, 100), 1), ((144, 144, 144), 1), ((256, 256, 256), 2), ((512, 512, 512), 2), ((64, 64, 64), 1), ((256, 320, 384), 4),
            ((2000, 4, 1000), 1), ((5000, 32, 32), 1)]
    for (s, ci), r in zip(full, rules(*(s for s, _ in full))):
        assert r["ci"] == ci, (s, r)


def test_row_parts_hold_whole_eighths_where_rows_still_fit(rules):
    shapes = [(200, 200, 1000), (256, 320, 384), (128, 192, 320), (150, 150, 400), (64, 64, 520), (100, 100, 100), (40, 40, 3000)]
    want = [(64, 4), (32, 8), (40, 6), (50, 5), (None, None), (25, 10), (64, 4)]
    for s, w, r in zip(shapes, want, rules(*shapes)):
        parts = -(-(-(-s[2] // r["vec"])) // r["bx"])
        assert w[0] is None or (r["bx"], r["by"]) == w, (s, r)
        assert r["by"] == 256 // r["bx"] and (parts == 1 or r["bx"] % 8 == 0 or (r["bx"] // 8 + 1) * 8 * r["by"] > 256), (s, r)
