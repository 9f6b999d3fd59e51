// oe_tiles.h -- the grid and the launch shapes of the Yee kernels.  Host code
// without HIP, so that the rules can be checked where there is no device.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>

namespace oe {

// Field block: one allocation of 6 arrays of N floats, E(x,y,z) then H(x,y,z).
// Coefficient block: 12 arrays of N floats, Ca(x,y,z) Cb(x,y,z) Da(x,y,z) Db(x,y,z).
struct Grid {
    int nx, ny, nz;
    size_t N;
};

// Yee kernel launch shape.  A work-group covers bx*V consecutive k of `by`
// rows (j) and marches along i over `ci` planes, keeping the i+1 (H update)
// or i-1 (E update) plane of the marched components in registers.
struct Tiles {
    int vec;  // 4: float4 accesses, 1: scalar
    int bx;   // lanes along k
    int by;   // rows along j; bx * by <= 256
    int ci;   // planes along i per work-group
};

// Whether a plane's byte offsets fit the float4 kernels' 32 bits (one row
// beyond either end included).
inline bool narrow_plane(const Grid& g) { return ((size_t)g.ny + 2) * g.nz < ((size_t)1 << 30); }

// Automatic tile choice: work-groups of at most 256 lanes, bx along k times
// by = 256 / bx rows of j, marching ci planes of i.
//
// bx: whole rows where a row's lanes fit (64 float4 lanes, 128 scalar ones,
// whose short segments cost more than idle lanes do), else the row cut into
// equal parts of at least 32 lanes that leave the fewest lanes idle.  A power
// of two left lanes idle on most grids: us per step at 100^3 (25 lanes)
// 32 / 25 lanes 13.9 / 11.9; 128x192x320 (80 lanes) 64 / 40 lanes 120 / 94;
// 256x320x384 (96 lanes) 64 / 32 lanes 466 / 426, with CPML 568 / 497; scalar
// 200x201x75 64 / 75 lanes 84.6 / 64.3.  Parts of a row are widened to a
// multiple of 8 lanes where as many rows still fit: a wave of 63 lanes' parts
// straddles two rows (200x200x1000, 63 / 64 lanes 632 / 596; 2000x18x2000 with
// CPML 1551 / 1428).
//
// ci: one plane up to 12 M cells, where more work-groups and a shorter chain
// of loads count (plain, us per step at ci 1 / 2 / 4: 64^3 8.0 / 9.3 / 12.2,
// 100^3 11.5 / 12.4 / 15.0, 160x144x120 37.0 / 39.2 / 38.2, 200^3 95.7 / 94.2 /
// 97.3); above, two planes, which reload half as many i +- 1 planes (256^3 198 /
// 186 / 184; 512^3 with CPML 2040 / 1950 / 1961), four where the row is cut
// into narrow blocks (256x320x384 with CPML 511 / 511 / 497).  A CPML grid's
// single launch takes one or two (oe_engine_run_batch).
// Scalar lanes, whose planes are cheaper than their start, take two
// (151x133x117 with CPML, ci 1 / 2 / 3: 82.5 / 75.0 / 81.0).
//
// Where a plane fills less than half of its work-groups' lanes, the start of a
// work-group costs more than the plane it works on, and the depth that pays
// grows as the square root of the work-groups (ci 1 or 2 / this: 100000x4x4
// 312 / 98, 100000x8x8 329 / 119, 20000x16x16 82 / 63, 1000x2x1000 30.5 / 28.7).
// No grid is cut into more than 2^23 work-groups of its tiles: a launch holds
// 2^32 lanes.
inline Tiles auto_tiles(const Grid& g, int vec_req) {
    Tiles t{};
    t.vec = vec_req == 1 || (g.nz % 4 != 0 && g.nz < 8) || !narrow_plane(g) ? 1 : 4;
    const int nzv = (g.nz + t.vec - 1) / t.vec;
    const int widest = t.vec == 4 ? 64 : 128;
    double best = 0.0;
    for (int n_kb = (nzv + widest - 1) / widest; n_kb <= nzv; ++n_kb) {
        const int bx = (nzv + n_kb - 1) / n_kb;
        if (best > 0.0 && (best >= 0.95 || bx < 32)) break;
        const double busy = (double)nzv * (256 / bx) / (256.0 * n_kb);
        if (busy > best) {
            best = busy;
            t.bx = bx;
        }
    }
    t.by = 256 / t.bx;
    const int n_kb = (nzv + t.bx - 1) / t.bx;
    if (n_kb > 1) t.bx = std::max(t.bx, 256 / t.by / 8 * 8);
    const int ci4 = g.N <= 12000000 ? 1 : (t.bx <= 32 && nzv > 64) ? 4 : 2;
    int ci = t.vec == 4 ? ci4 : 2;
    const double blocks = (double)n_kb * ((g.ny + t.by - 1) / t.by);  // work-groups of a plane
    if ((double)nzv * g.ny < 128.0 * blocks) ci = std::max(ci, (int)(std::sqrt(blocks * g.nx) / 16));
    ci = std::max(ci, (int)std::ceil(blocks * g.nx / (1 << 23)));
    t.ci = std::min(g.nx, ci);
    return t;
}

// Cells of a row that a lane of the sweep's own launches (structures without a
// single launch) takes; z_aligned: the CPML z slabs, if any, hold whole float4s.
inline int sweep_lanes(const Grid& g, bool z_aligned) { return g.nz % 4 == 0 && z_aligned && narrow_plane(g) ? 4 : 1; }

}  // namespace oe
