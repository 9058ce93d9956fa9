// The tiles of a resident 2D run and the rim cells its blocks take from each
// other; host code as well, for the check of the exchange.
#pragma once
#include <algorithm>

#include "seis_internal.hpp"

namespace seis {
namespace {

// Tiles of a grid for one instantiation: nbz x nbx blocks of cores CZ x CX.
struct Tiling {
    int nbz = 0, nbx = 0, cz = 0, cx = 0;
};
// The fewest rows of tiles, evenly high, then as many columns as the chip has
// CUs for, but no core narrower than kMinCX.
constexpr int kMinCX = 4;
inline Tiling tiling(const Layout &g, int cols, int ncu) {
    Tiling t;
    const int H = g.H, nz = g.NZ + 2 * H, nx = g.NX + 2 * H, czm = 64 - 2 * H, cxm = cols - 2 * H;
    ncu = ncu / 8 * 8;   // the launch rounds the number of blocks up to 8
    if (cxm < 1 || ncu < 8) return t;
    t.nbz = (nz + czm - 1) / czm;
    t.cz = std::max((nz + t.nbz - 1) / t.nbz, 2 * H + 1);
    t.nbz = (nz + t.cz - 1) / t.cz;
    if (t.nbz > ncu) return Tiling();
    t.cx = std::max(kMinCX, (nx + ncu / t.nbz - 1) / (ncu / t.nbz));
    if (t.cx > cxm) return Tiling();
    t.nbx = (nx + t.cx - 1) / t.cx;
    return t;
}

// cells of the rim that a block takes from others: z sides, x sides, corners
SEIS_HD constexpr int rim_cells(int H, int CX, int CZ) { return 4 * H * CX + 4 * H * CZ + 4 * H * H; }

// A block whose core holds halo cells alone takes no rim cells: it updates
// nothing, and nobody takes words from it, so that nobody would wait until it has
// read theirs.
template <int H>
SEIS_HD inline bool halo_block(const Layout &g, int CZ, int CX, int rz0, int rx0) {
    const int z = rz0 + 2 * H, x = rx0 + 2 * H;   // the core's first cell
    return z >= g.NZ || z + CZ <= 0 || x >= g.NX || x + CX <= 0;
}
// Its place in the grid of a neighbour's cell whose words change with the
// neighbour's steps (the grid's cell closest to the core, among the outer 2H of
// the neighbour's), else -1.
template <int H>
SEIS_HD inline int pulse_cell(const Layout &g, int CZ, int CX, int rz0, int rx0) {
    if (!halo_block<H>(g, CZ, CX, rz0, rx0)) return -1;
    const int z = rz0 + 2 * H, x = rx0 + 2 * H;
    return (int)g.idx(z < 0 ? 0 : z < g.NZ ? z : g.NZ - 1, 0, x < 0 ? 0 : x < g.NX ? x : g.NX - 1);
}

// The q-th rim cell of a block with its region at (rz0, rx0): its LDS cell and
// its place in the grid, -1 if there is none or it never changes (images: the
// image rows above the free surface do).
template <int H, int RZ>
SEIS_HD inline void rim_cell(const Layout &g, int images, int CZ, int CX, int rz0, int rx0, int q,
                             int &rl, int &ri) {
    int lx = 0, lz = 0;
    bool in = !halo_block<H>(g, CZ, CX, rz0, rx0);
    const int nz = 4 * H * CX, nx = 4 * H * CZ;
    if (q < nz) {
        lz = q % (4 * H);
        lx = 2 * H + q / (4 * H);
        if (lz >= 2 * H) lz += CZ;
    } else if ((q -= nz) < nx) {
        lz = 2 * H + q % CZ;
        lx = q / CZ;
        if (lx >= 2 * H) lx += CX;
    } else if ((q -= nx) < 4 * H * H) {
        lz = H + q % (2 * H);
        lx = H + q / (2 * H);
        if (lz >= 2 * H) lz += CZ;
        if (lx >= 2 * H) lx += CX;
    } else {
        in = false;
    }
    const int zz = rz0 + lz, xx = rx0 + lx;
    in = in && zz >= (images ? -H : 0) && zz < g.NZ && xx >= 0 && xx < g.NX;
    rl = lx * RZ + lz;
    ri = in ? (int)g.idx(zz, 0, xx) : -1;
}

}  // namespace
}  // namespace seis
