// Host check of the exchange of resident 2D runs (seis::tiling, seis::rim_cell):
// a block overwrites a word two steps after it published it, having taken words
// of the step between from every block whose rim the word lies in.  That holds if
// block A takes cells of block B exactly if B takes cells of A, and every word
// that is waited for is one that its owner publishes (the outer 2H cells of its
// core).  Blocks of halo cells neither take nor are waited for.  And the pause
// after a run that gave up (seis::RunRest).  Built and run by test_lib_cpu.py.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>

#include "resident_tiles.hpp"

static int bad = 0, grids = 0;
static long halo_blocks = 0;

template <int H>
static void check(int NZ, int NX, int cols, int ncu, int images) {
    using namespace seis;
    Layout g = make_layout(2, NZ, 1, NX, H, 4);
    const Tiling t = tiling(g, cols, ncu);
    if (!t.nbz) return;
    ++grids;
    const int nb = t.nbz * t.nbx;
    if (nb > ncu) ++bad;
    std::vector<std::set<int>> takes(nb);
    for (int b = 0; b < nb; ++b) {
        const int bz = b % t.nbz, bx = b / t.nbz;
        const int rz0 = -H + bz * t.cz - 2 * H, rx0 = -H + bx * t.cx - 2 * H;
        const int z0 = rz0 + 2 * H, x0 = rx0 + 2 * H;
        // a block of halo cells watches a word that its neighbour publishes
        const bool halo = z0 >= NZ || z0 + t.cz <= 0 || x0 >= NX || x0 + t.cx <= 0;
        const int pulse = pulse_cell<H>(g, t.cz, t.cx, rz0, rx0);
        if (halo != (pulse >= 0)) ++bad;
        if (halo) {
            const int zz = pulse % (int)g.ldz - g.ZO, xx = pulse / (int)g.ldz - H;
            const int cz = (zz + H) % t.cz, cx = (xx + H) % t.cx;
            if (zz < 0 || zz >= NZ || xx < 0 || xx >= NX ||
                !(cz < 2 * H || cz >= t.cz - 2 * H || cx < 2 * H || cx >= t.cx - 2 * H))
                ++bad;
            ++halo_blocks;
        }
        for (int q = 0; q < rim_cells(H, t.cx, t.cz); ++q) {
            int rl, ri;
            rim_cell<H, 64 + 2 * H>(g, images, t.cz, t.cx, rz0, rx0, q, rl, ri);
            if (ri < 0) continue;
            const int zz = ri % (int)g.ldz - g.ZO, xx = ri / (int)g.ldz - H;
            const int oz = (zz + H) / t.cz, ox = (xx + H) / t.cx, o = ox * t.nbz + oz;
            const int cz = (zz + H) % t.cz, cx = (xx + H) % t.cx;   // in the owner's core
            const bool ez = cz < 2 * H || cz >= t.cz - 2 * H, ex = cx < 2 * H || cx >= t.cx - 2 * H;
            // (image rows are published for the outer columns)
            if (o == b || xx < 0 || xx >= NX || zz >= NZ || !(ex || (ez && zz >= 0))) ++bad;
            takes[b].insert(o);
        }
    }
    int one_way = 0;
    for (int b = 0; b < nb; ++b)
        for (int o : takes[b])
            if (!takes[o].count(b)) ++one_way;
    if (one_way) {
        if (!bad)
            std::printf("%d x %d, H %d, %d columns, %d CUs: %d blocks wait for one that does not "
                        "wait for them\n", NZ, NX, H, cols, ncu, one_way);
        ++bad;
    }
}

template <int H>
static void sweep(std::mt19937 &rng) {
    auto size = [&](int lo, int hi) {
        return lo + (int)(rng() % (unsigned)(hi - lo + 1));
    };
    for (int cols : {16, 32, 48, 80})
        for (int k = 0; k < 60; ++k) {
            const int ncu = k % 4 ? 256 : 64, top = k % 2 ? 600 : 150;
            check<H>(size(2 * H, top), size(2 * H, 3 * top), cols, ncu, k % 3 == 0);
        }
    check<H>(100, 100, 16, 256, 0);
    check<H>(211, 397, 16, 256, 1);
}

// The pause after a run that gave up: a hundred waits, then runs again.
static void check_rest() {
    using namespace std::chrono;
    const auto t = seis::RunRest::clock::now();
    seis::RunRest r;
    if (!r.over(t)) ++bad;
    r.set_wait(5);
    if (!r.over(t)) ++bad;
    r.begin(t);
    if (r.over(t) || r.over(t + milliseconds(499)) || !r.over(t + milliseconds(500))) ++bad;
    r.set_wait(0);
    r.begin(t);
    if (!r.over(t)) ++bad;
}

int main() {
    check_rest();
    std::mt19937 rng(7);
    sweep<1>(rng);
    sweep<2>(rng);
    sweep<3>(rng);
    sweep<4>(rng);
    sweep<5>(rng);
    sweep<6>(rng);
    std::printf("%d grids, %ld blocks of halo cells alone, %d faults\n", grids, halo_blocks, bad);
    return bad || grids < 300 || halo_blocks < 100;
}
