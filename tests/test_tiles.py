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
