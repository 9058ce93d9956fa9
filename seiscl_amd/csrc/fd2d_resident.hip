// 2D runs resident on the chip: one launch makes all the steps of a run.
//
// A 2D step of the ordinary kernels is three or four dependent launches
// (sources and receivers, velocities, stresses, surface) of 3-8 us each,
// however small the grid: kernel start, a trip to memory past the L2s, which a
// kernel boundary empties, and the write-back at its end.  The state of a 2D
// grid fits the registers and LDS of the 256 CUs, so here every block keeps a
// tile of it for the whole run: wavefields in LDS, what is private to a cell
// (coefficients, memory variables, CPML memory) in registers.  Per step a
// block
//   1. adds the sources,
//   2. updates the velocities of its core and of a rim H cells wide (the rim
//      twice, by its owner and here: the same operations on the same values),
//   3. updates the stresses of its core and applies the free surface,
//   4. records its receivers,
//   5. publishes the stresses of its core's outer 2H cells and takes the
//      2H cells around its core from the other blocks.
// That is one exchange per step.  Velocities and CPML memory of the rim are
// never exchanged: they start equal to the owner's and stay so.
//
// Exchange: a cell's values and the number of their step travel together in
// 64-bit words, stored and loaded with relaxed agent-scope atomics (a 64-bit
// access is single-copy atomic, so a word that carries the step's number carries
// the step's value: no fence, no flag).  The pressure is one word with 32 bits
// of the number; three stresses are two words with 16 bits each.  Words lie at
// the cell's place in the padded grid, in two buffers that steps use in turn
// and that are cleared before the run.  A block overwrites a buffer two steps
// later, after it took the words of the step between from every block it
// shares a rim with, which those published after they had taken this buffer's.
// Halo cells of the grid do not change and are not exchanged, the image rows
// apart; a block whose core holds nothing else takes no words, since it gives
// none that the others would wait for (resident_tiles.hpp).
//
// Every block must be on the chip at once: there is at most one per CU, and the
// host makes one such run at a time on a GPU.  Kernels of other streams end and
// make room.  Where another program holds CUs for good, a block that waits
// longer than a.patience (wall_clock64 ticks) gives up, so the grid ends in any
// case.  Results are written only once every block has made its last step: the
// last one to get there sets the run's state to "complete", a block that gives
// up sets it to "failed", whichever comes first, and every block obeys it.  A
// failed run leaves the model's state as it was, and the caller makes the steps
// with the ordinary kernels.  (A cooperative launch goes through a queue of its
// own: with a second context in use, changing between it and the context's
// stream took 1.3 ms per run.)
//
// One wave holds 64 consecutive z of N consecutive x of the core and its rim:
// LDS rows are read without bank conflicts, the x-derivatives of a lane's N
// cells share a window of N + 2H - 1 values, and what depends on x alone is
// uniform.  The outer H cells of the region have no lane; they are only read.
//
// The domain is the padded grid, [-H, N + H) per axis: halo cells are loaded
// and stored like the others, and not updated or exchanged, except for the image
// rows of the free surface.
//
// What bounds a step is the exchange (a store and a load past the L2s, 1.5-2 us)
// and, from about 1000 cells per CU on, the tile's arithmetic and LDS reads with
// the barriers between them (at 2100 and 3500 cells per CU the VALUs are busy 44
// and 41 % of the time, the LDS 31 and 38 %).  Measured on MI355X, us
// per step, step kernels (replayed graphs) -> this kernel:
//                     100 x 100    200 x 400    433 x 1217   600 x 1500
//   elastic FD4       9.5 -> 2.6   9.8 -> 2.9   13.3 -> 6.4  19.9 -> 13.1
//   elastic FD8       9.8 -> 3.4   9.8 -> 3.6   15.2 -> 8.3  22.5 -> 17.9
//   L = 1, FD4        13.3 -> 2.7  14.4 -> 3.0  24.3 -> 6.8  not covered
//   acoustic FD8      8.5 -> 2.4   8.6 -> 2.4   11.5 -> 4.5  14.3 -> 6.1
// (L = 1 with a free surface.)  Stepping tiles with a halo of 2 H K cells for K
// steps per launch, without an exchange, costs 10 us to load a 64 x 32 region,
// about 18 KB per us and CU, and wins on no FD order above 2.
//
// Arithmetic: the cell updates of fd_kernels.hip, term by term.
#include <hip/hip_runtime.h>

#include "resident2d.hpp"

namespace seis {
namespace {

// ACOUSTIC: fields vx, vz, p (else vx, vz, sxx, szz, sxz); L Maxwell bodies
// (elastic case only).  NW waves, N columns of x per lane.
template <int H, bool ACOUSTIC, int L, int NW, int N>
__global__ __launch_bounds__(64 * NW) void k_resident2d(Resident2D a) {
    // the region: 64 + 2H rows of z, NW N + 2H columns
    constexpr int RZ = 64 + 2 * H, RX = NW * N + 2 * H, NF = ACOUSTIC ? 3 : 5, FS = RX * RZ;
    constexpr int NP = ACOUSTIC ? 4 : 8, HP = NP / 4, NC = ACOUSTIC ? 3 : L ? 8 : 5;
    constexpr int LS = L > 0 ? L : 1;
    constexpr int NE = resident_values(ACOUSTIC);   // exchanged fields, the last of NF
    // rim cells per thread
    constexpr int MR = (rim_cells(H, RX - 4 * H, RZ - 4 * H) + 64 * NW - 1) / (64 * NW);
    static_assert(RX * RZ <= 8192, "rlist packing");
    __shared__ float lds[NF * FS];
    __shared__ int rlist[kResidentMaxRec];             // receiver << 13 | cell
    __shared__ float xprof[6 * (kMaxNab + 1)];
    __shared__ int scell[kResidentMaxSrc], sfield[kResidentMaxSrc];
    __shared__ float samp[kResidentMaxSrc];
    __shared__ int rcount, dead, verdict, pulse;

    unsigned tile;
    xcd_tile(a.ntile, tile);
    if (tile >= a.ntile) return;
    const Layout &g = a.g;
    const int NZ = g.NZ, NX = g.NX, NAB = a.nab;
    const int lane = threadIdx.x, w = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int tid = w * 64 + lane;
    const int CZ = a.cz, CX = a.cx;
    const int bz = tile % a.nbz, bx = tile / a.nbz;
    // region origin; the core starts at (2H, 2H), lane 0 and column 0 at (H, H)
    const int rz0 = -H + bz * CZ - 2 * H, rx0 = -H + bx * CX - 2 * H;
    const int z = rz0 + H + lane, x0 = rx0 + H + w * N;
    const bool zpad = z >= -H && z < NZ + H, zin = z >= 0 && z < NZ;
    const bool core_z = lane >= H && lane < H + CZ, rim_z = lane < CZ + 2 * H;
    const bool edge_z = core_z && (lane < 3 * H || lane >= CZ - H);

    if (tid == 0) {
        rcount = 0;
        dead = 0;
        pulse = pulse_cell<H>(g, CZ, CX, rz0, rx0);
    }
    float *F = lds + (H + w * N) * RZ + H + lane;   // the lane's first cell of field 0
    float co[NC][N], ps[NP][N], mv[3 * LS][N];
    const bool cpml = a.abs_type == 1;
    const bool zbot = z > NZ - NAB - 1;
    const bool pz = cpml && zin && (zbot || (!a.freesurf && z < NAB));
    const int kz = zbot ? z - NZ + 2 * NAB : z;
    // the lane's columns: in the grid and updated (velocities; stresses),
    // in the core, in an x strip, among the core's outer 2H columns
    unsigned mvel = 0, mstr = 0, mcore = 0, mpx = 0, medge = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int c = w * N + j, x = x0 + j;
        const bool in = x >= 0 && x < NX, core = c >= H && c < H + CX;
        mvel |= (unsigned)(in && c < CX + 2 * H) << j;
        mstr |= (unsigned)(in && core) << j;
        mcore |= (unsigned)(core && x < NX + H) << j;
        medge |= (unsigned)(core && (c < 3 * H || c >= CX - H)) << j;
        mpx |= (unsigned)(cpml && in && (x < NAB || x > NX - NAB - 1)) << j;
    }
    mvel = __builtin_amdgcn_readfirstlane(mvel);
    mstr = __builtin_amdgcn_readfirstlane(mstr);
    mcore = __builtin_amdgcn_readfirstlane(mcore);
    mpx = __builtin_amdgcn_readfirstlane(mpx);
    medge = __builtin_amdgcn_readfirstlane(medge);
    Prof zp = {1, 0, 0, 1, 0, 0};
    // the region's fields
    for (int q = tid; q < FS; q += 64 * NW) {
        const int zz = rz0 + q % RZ, xx = rx0 + q / RZ;
        const bool in = zz >= -H && zz < NZ + H && xx >= -H && xx < NX + H;
        const long i = in ? g.idx(zz, 0, xx) : 0;
#pragma unroll
        for (int e = 0; e < NF; ++e) lds[e * FS + q] = in ? a.f[e][i] : 0.0f;
    }
    {
        const int zc = min(max(z, -H), NZ + H - 1);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int xc = min(max(x0 + j, -H), NX + H - 1);
            const long i = g.idx(zc, 0, xc);
#pragma unroll
            for (int q = 0; q < NC; ++q) co[q][j] = a.co[q][i];
#pragma unroll
            for (int q = 0; q < 3 * L; ++q) mv[q][j] = a.m[q / LS][(q % LS) * g.nfield + i];
#pragma unroll
            for (int q = 0; q < NP; ++q) ps[q][j] = 0;
        }
        if (__any(pz)) {
            const int kc = pz ? kz : 0;
            zp = prof_load(a.cpml + 12 * 2 * NAB, 2 * NAB, pz && zbot ? 2 * NAB - kz : kc,
                           pz && zbot ? 2 * NAB - 1 - kz : kc);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const long iz = (long)min(max(x0 + j, 0), NX - 1) * 2 * NAB + kc;
#pragma unroll
                for (int q = 0; q < NP; ++q)
                    if ((q / HP) % 2 == 0) ps[q][j] = a.p[q][iz];
            }
        }
        if (mpx) {
            const int zi = min(max(z, 0), NZ - 1);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (!(mpx >> j & 1)) continue;
                const int x = x0 + j, ii = x < NAB ? x : x - NX + 2 * NAB;
#pragma unroll
                for (int q = 0; q < NP; ++q)
                    if ((q / HP) % 2 == 1) ps[q][j] = a.p[q][(long)ii * NZ + zi];
            }
        }
        if (cpml)
            for (int q = tid; q < 6 * (NAB + 1); q += 64 * NW)
                xprof[q] = a.cpml[(q % 6) * 2 * NAB + min(q / 6, 2 * NAB - 1)];
    }
    __syncthreads();
    // sources of the region, in order (wave 0: lane q feeds source q), and
    // receivers of the core
    int ns = 0;
    const float *ssrc = nullptr;
    float snext = 0;
    {
        int cell = -1, sz = 0, sx = 0;
        if (lane < a.s.nsrc) cell = a.s.src_cell[lane];
        bool here = cell >= 0;
        if (here) {
            sx = cell / (int)g.ldz - g.H - rx0;
            sz = cell % (int)g.ldz - g.ZO - rz0;
            here = sx >= 0 && sx < CX + 4 * H && sz >= 0 && sz < CZ + 4 * H;
        }
        const unsigned long long mask = __ballot(here);
        ns = __popcll(mask);
        if (w == 0) {
            if (here) {
                const int k = __popcll(mask & ((1ull << lane) - 1));
                scell[k] = sx * RZ + sz;
                sfield[k] = source_field<ACOUSTIC>(a.s.src_type[lane]);
                samp[k] = __int_as_float(lane);
            }
            __builtin_amdgcn_wave_barrier();
            if (lane < ns) {
                ssrc = a.s.src + (long)__float_as_int(samp[lane]) * a.NT;
                snext = ssrc[a.t0];
            }
        }
    }
    for (int r = tid; r < a.s.nrec; r += 64 * NW) {
        const int cell = a.s.rec_cell[r];
        if (cell < 0) continue;
        const int lx = cell / (int)g.ldz - g.H - rx0, lz = cell % (int)g.ldz - g.ZO - rz0;
        if (lx < 2 * H || lx >= 2 * H + CX || lz < 2 * H || lz >= 2 * H + CZ) continue;
        rlist[atomicAdd(&rcount, 1)] = r << 13 | (lx * RZ + lz);
    }
    // the rim cells this thread takes
    int rl[MR], ri[MR];
#pragma unroll
    for (int e = 0; e < MR; ++e)
        rim_cell<H, RZ>(g, a.freesurf, CZ, CX, rz0, rx0, tid + e * 64 * NW, rl[e], ri[e]);
    __syncthreads();
    const int nr = rcount;
    const float *hc = a.hc;

    const int x0_ = x0, z_ = z;
    for (int k = 0; k < a.nsteps; ++k) {
        const int t = a.t0 + k;
        // what follows from a lane's place is computed in every step: kept over
        // the loop it takes more registers than the state does
        int x0 = x0_, z = z_;
        asm volatile("" : "+s"(x0), "+v"(z));
        const unsigned tag = k + 1;
        Word *X = a.xch + (size_t)(tag & 1) * resident_nwords(NE) * g.nfield;
        const bool last = k + 1 == a.nsteps;
        if (ns) {
            if (w == 0) {
                if (lane < ns) {
                    samp[lane] = snext;
                    if (k + 1 < a.nsteps) snext = ssrc[t + 1];
                }
                __builtin_amdgcn_wave_barrier();
                if (lane == 0) {
                    float *B = lds;
                    for (int q = 0; q < ns; ++q) {
                        const int c = scell[q], f = sfield[q];
                        const float amp = a.DT * samp[q];
                        if (f >= 0) {
                            B[f * FS + c] = B[f * FS + c] + amp;
                            continue;
                        }
                        if constexpr (!ACOUSTIC)
                            if (f == kSourceNormal)
                                for (int e = 2; e < 4; ++e)
                                    B[e * FS + c] =
                                        (float)((double)B[e * FS + c] + (double)amp / 2.0);
                    }
                }
            }
            __syncthreads();
        }
        if (a.hist && core_z && zin) {
            // the state after the sources, for an adjoint run
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int x = x0 + j;
                if (!(mstr >> j & 1)) continue;
                float *h = a.hist + (long)k * NF * g.nfield + g.idx(z, 0, x);
#pragma unroll
                for (int q = 0; q < NF; ++q) h[q * g.nfield] = F[q * FS + j * RZ];
            }
        }
        // velocities of the core and its rim
        if (mvel) {
            float da[N], db[N];
            dx<H, N, true, RZ>(F + 2 * FS, hc, da);                            // sxx_x or p_x
            if constexpr (!ACOUSTIC) dx<H, N, false, RZ>(F + 4 * FS, hc, db);   // sxz_x
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int x = x0 + j;
                if (!(mvel >> j & 1)) continue;
                float *f = F + j * RZ;
                const bool px = mpx >> j & 1;
                const int ii = x < NAB ? x : NX - x, ih = x < NAB ? x : NX - 1 - x;
                float vx, vz;
                if constexpr (ACOUSTIC) {
                    float p_z = dz<H, true>(f + 2 * FS, hc), p_x = da[j];
                    if (pz) pmlh(p_z, ps[0][j], zp);
                    if (px) pmlh(p_x, ps[1][j], prof_x(xprof, ii, ih));
                    vx = f[0] + (p_x * co[0][j]);
                    vz = f[FS] + (p_z * co[1][j]);
                } else {
                    float szz_z = dz<H, true>(f + 3 * FS, hc), sxz_z = dz<H, false>(f + 4 * FS, hc);
                    float sxx_x = da[j], sxz_x = db[j];
                    if (pz) {
                        pmlf(sxz_z, ps[0][j], zp);
                        pmlh(szz_z, ps[1][j], zp);
                    }
                    if (px) {
                        const Prof xp = prof_x(xprof, ii, ih);
                        pmlh(sxx_x, ps[2][j], xp);
                        pmlf(sxz_x, ps[3][j], xp);
                    }
                    vx = f[0] + ((sxx_x + sxz_z) * co[0][j]);
                    vz = f[FS] + ((szz_z + sxz_x) * co[1][j]);
                }
                if (a.abs_type == 2 && zin) {
                    const float *tp = a.taper;
                    if ((ACOUSTIC || !a.freesurf) && z < NAB) { vx *= tp[z]; vz *= tp[z]; }
                    if (z > NZ - NAB - 1) { vx *= tp[NZ - z - 1]; vz *= tp[NZ - z - 1]; }
                    if (x < NAB) { vx *= tp[x]; vz *= tp[x]; }
                    if (x > NX - NAB - 1) { vx *= tp[NX - x - 1]; vz *= tp[NX - x - 1]; }
                }
                if (zin && rim_z) {
                    f[0] = vx;
                    f[FS] = vz;
                }
            }
        }
        __syncthreads();
        // stresses of the core and the free surface
        if (mstr) {
            float da[N], db[N];
            dx<H, N, false, RZ>(F, hc, da);                                // vxx
            if constexpr (!ACOUSTIC) dx<H, N, true, RZ>(F + FS, hc, db);   // vzx
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int x = x0 + j;
                if (!(mstr >> j & 1)) continue;
                float *f = F + j * RZ;
                const bool px = mpx >> j & 1;
                const int ii = x < NAB ? x : NX - x, ih = x < NAB ? x : NX - 1 - x;
                float vxx = da[j], vzz = dz<H, false>(f + FS, hc);
                if constexpr (ACOUSTIC) {
                    if (pz) pmlf(vzz, ps[2][j], zp);
                    if (px) pmlf(vxx, ps[3][j], prof_x(xprof, ii, ih));
                    float p = f[2 * FS];
                    p += (co[2][j] * (vxx + vzz));
                    if (a.abs_type == 2 && zin) {
                        const float *tp = a.taper;
                        if (z < NAB) p *= tp[z];
                        if (z > NZ - NAB - 1) p *= tp[NZ - z - 1];
                        if (x < NAB) p *= tp[x];
                        if (x > NX - NAB - 1) p *= tp[NX - x - 1];
                    }
                    if (zin && core_z) {
                        f[2 * FS] = p;
                        if (!last && (edge_z || (medge >> j & 1)))
                            put_cell<1>(X, 0, g.idx(z, 0, x), &p, tag);
                    }
                } else {
                    float vxz = dz<H, true>(f, hc), vzx = db[j];
                    if (pz) {
                        pmlh(vxz, ps[4][j], zp);
                        pmlf(vzz, ps[5][j], zp);
                    }
                    if (px) {
                        const Prof xp = prof_x(xprof, ii, ih);
                        pmlf(vxx, ps[6][j], xp);
                        pmlh(vzx, ps[7][j], xp);
                    }
                    float sxx = f[2 * FS], szz = f[3 * FS], sxz = f[4 * FS];
                    const float DT2 = a.DT2;
                    float gg, ff, d = 0, e = 0;
                    if constexpr (L == 0) {
                        gg = co[2][j];
                        ff = 2.0f * co[3][j];
                        sxz += (co[4][j] * (vxz + vzx));
                        sxx += (gg * (vxx + vzz)) - (ff * vzz);
                        szz += (gg * (vxx + vzz)) - (ff * vxx);
                    } else {
                        gg = co[2][j];
                        ff = co[3][j];
                        d = co[4][j];
                        e = co[5][j];
                        const float fipkp = co[6][j], dipkp = co[7][j];
                        float mxz = 0, mxx = 0, mzz = 0;
#pragma unroll
                        for (int l = 0; l < L; ++l) {
                            mxz += mv[2 * L + l][j];
                            mxx += mv[l][j];
                            mzz += mv[L + l][j];
                        }
                        const float lsxz = (fipkp * (vxz + vzx)) + (DT2 * mxz);
                        const float lsxx = ((gg * (vxx + vzz)) - (ff * vzz)) + (DT2 * mxx);
                        const float lszz = ((gg * (vxx + vzz)) - (ff * vxx)) + (DT2 * mzz);
                        mxz = mxx = mzz = 0;
#pragma unroll
                        for (int l = 0; l < L; ++l) {
                            const float b = a.bl[l], c = a.cl[l], et = a.eta[l];
                            float &rxz = mv[2 * L + l][j], &rxx = mv[l][j], &rzz = mv[L + l][j];
                            rxz = b * (rxz * c - et * (dipkp * (vxz + vzx)));
                            rxx = b * (rxx * c - et * ((e * (vxx + vzz)) - (d * vzz)));
                            rzz = b * (rzz * c - et * ((e * (vxx + vzz)) - (d * vxx)));
                            mxz += rxz;
                            mxx += rxx;
                            mzz += rzz;
                        }
                        sxz += lsxz + (DT2 * mxz);
                        sxx += lsxx + (DT2 * mxx);
                        szz += lszz + (DT2 * mzz);
                    }
                    if (a.abs_type == 2 && zin) {
                        const float *tp = a.taper;
                        if (!a.freesurf && z < NAB) { sxx *= tp[z]; szz *= tp[z]; sxz *= tp[z]; }
                        if (z > NZ - NAB - 1) {
                            const float q = tp[NZ - z - 1];
                            sxx *= q; szz *= q; sxz *= q;
                        }
                        if (x < NAB) { sxx *= tp[x]; szz *= tp[x]; sxz *= tp[x]; }
                        if (x > NX - NAB - 1) {
                            const float q = tp[NX - x - 1];
                            sxx *= q; szz *= q; sxz *= q;
                        }
                    }
                    if (a.bnd && zin && core_z) {
                        // boundary shell of the step, before the surface
                        const long m = a.sh.inject(z + H, 0, x + H);
                        if (m >= 0) {
                            float *b = a.bnd + (long)t * NF * a.sh.n + m;
                            b[0] = f[0];
                            b[a.sh.n] = f[FS];
                            b[2 * a.sh.n] = sxx;
                            b[3 * a.sh.n] = szz;
                            b[4 * a.sh.n] = sxz;
                        }
                    }
                    if (a.freesurf && core_z && z >= 0 && z <= H) {
                        // image method (src/surface2D.cl): the lane of z = 0
                        // holds the derivatives and memory variables it needs
                        if (z == 0) {
                            szz = 0;
                            float h = -((gg - ff) * (gg - ff) * (vxx) / gg) - ((gg - ff) * vzz);
                            if constexpr (L == 0) {
                                sxx = sxx + 1.0f * h;
                            } else {
                                float sump = 0;
#pragma unroll
                                for (int l = 0; l < L; ++l) {
                                    mv[L + l][j] = 0;
                                    sump += mv[l][j];
                                }
                                h += -DT2 * sump;
                                const float sxxv = sxx + 1.0f * h;
                                sump = 0;
#pragma unroll
                                for (int l = 0; l < L; ++l) {
                                    const double b =
                                        (double)a.eta[l] / (1.0 + ((double)a.eta[l] * 0.5));
                                    const float bb = (float)b;
                                    const float q =
                                        (float)((double)bb *
                                                ((double)(d - e) * ((double)(ff / gg) - 1.0) *
                                                     (double)vxx -
                                                 (double)((d - e) * vzz)));
                                    mv[l][j] = mv[l][j] + 1.0f * q;
                                    sump += mv[l][j];
                                }
                                sxx = sxxv + 1.0f * (DT2 * sump);
                            }
                        }
                        if (z >= 1) f[3 * FS - 2 * z] = -szz;
                        if (z < H) f[4 * FS - 2 * z - 1] = -sxz;
                    }
                    if (zin && core_z) {
                        f[2 * FS] = sxx;
                        f[3 * FS] = szz;
                        f[4 * FS] = sxz;
                        if (!last && (edge_z || (medge >> j & 1))) {
                            const float v[3] = {sxx, szz, sxz};
                            put_cell<3>(X, g.nfield, g.idx(z, 0, x), v, tag);
                        }
                    }
                }
            }
        }
        __syncthreads();
        if (a.freesurf && !last && mstr && core_z && z >= -H && z < 0) {
            // image rows of the core's outer columns
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (!(mstr & medge & 1u << j)) continue;
                if constexpr (!ACOUSTIC) {
                    const float *f = F + j * RZ, v[3] = {f[2 * FS], f[3 * FS], f[4 * FS]};
                    put_cell<3>(X, g.nfield, g.idx(z, 0, x0 + j), v, tag);
                }
            }
        }
        if (nr) {
            const float *B = lds;
            float *out = a.s.out + (long)t * a.nout * a.s.nrec;
            for (int q = tid; q < nr * a.nout; q += 64 * NW) {
                const int e = rlist[q % nr], o = q / nr, c = e & 8191, code = a.code[o];
                float v;
                if constexpr (ACOUSTIC) {
                    v = B[(code == O_VX ? 0 : code == O_VZ ? 1 : 2) * FS + c];
                } else if (code == O_P) {
                    const float sm = B[2 * FS + c] + B[3 * FS + c];
                    v = (float)((double)sm / 2.0);
                } else {
                    v = B[(code == O_VX    ? 0
                           : code == O_VZ  ? 1
                           : code == O_SXX ? 2
                           : code == O_SZZ ? 3
                                           : 4) * FS + c];
                }
                out[(long)o * a.s.nrec + (e >> 13)] = v * a.unscale[o];
            }
        }
        if (last) break;
        const bool ok = take_rim<NE, MR>(X, g.nfield, tag, a.patience, ri, [&](int e, const float *u) {
#pragma unroll
            for (int q = 0; q < NE; ++q) lds[(2 + q) * FS + rl[e]] = u[q];
        });
        if (!ok && lane == 0) dead = 1;
        __syncthreads();
        if (dead) break;
    }

    // every block's last step is made, or the run has failed
    if (tid == 0)
        verdict = agree(a.sync, a.failed, (int)a.ntile, dead, a.patience,
                        pulse < 0 ? nullptr : a.xch + pulse);
    __syncthreads();
    if (verdict != 1) return;

    // the core, halo cells of the grid included
    if (!core_z || !zpad) return;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int x = x0 + j;
        if (!(mcore >> j & 1)) continue;
        const long i = g.idx(z, 0, x);
#pragma unroll
        for (int q = 0; q < NF; ++q) a.f[q][i] = F[q * FS + j * RZ];
        if (!zin || x < 0 || x >= NX) continue;
#pragma unroll
        for (int q = 0; q < 3 * L; ++q) a.m[q / LS][(q % LS) * g.nfield + i] = mv[q][j];
        const bool px = mpx >> j & 1;
        const int ii = x < NAB ? x : x - NX + 2 * NAB;
        const long iz = (long)x * 2 * NAB + kz, ix = (long)ii * NZ + z;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const bool isz = (q / HP) % 2 == 0;
            if (isz ? pz : px) a.p[q][isz ? iz : ix] = ps[q][j];
        }
    }
}

template <int H, bool ACOUSTIC, int L, int NW, int N>
bool run_resident(Resident2D &a, int ncu, hipStream_t st, int &err) {
    const Tiling t = tiling(a.g, NW * N, ncu);
    if (!t.nbz) return false;
    a.cz = t.cz;
    a.cx = t.cx;
    a.nbz = t.nbz;
    a.ntile = (unsigned)(t.nbz * t.nbx);
    if (!st) return true;
    hipLaunchKernelGGL((k_resident2d<H, ACOUSTIC, L, NW, N>), dim3((a.ntile + 7) / 8 * 8), dim3(64, NW), 0, st, a);
    err = (int)hipGetLastError();
    return true;
}

// The smallest region that covers the grid.  The lines lie where the next
// instantiation, or the step kernels, are faster (us per step, resident against
// step kernels): with one Maxwell body 16 x 3 columns lose to 8 x 6 from FD order 8
// on (433 x 1217: 11.2 against 10.5; FD4 6.8 against 8.7); on 80 columns a Maxwell
// body spills, and the step kernels take those grids (600 x 1500, two bodies FD4:
// 32.8 against 28.0, one body FD8: 35.0 against 32.7).
template <int H>
bool dispatch(Resident2D &a, int nd_case, int ncu, hipStream_t st, int &err) {
    if (nd_case == 22)
        return run_resident<H, true, 0, 16, 1>(a, ncu, st, err) ||
               run_resident<H, true, 0, 16, 2>(a, ncu, st, err) ||
               run_resident<H, true, 0, 16, 3>(a, ncu, st, err) ||
               run_resident<H, true, 0, 16, 5>(a, ncu, st, err);
    switch (a.L) {
        case 0:
            return run_resident<H, false, 0, 16, 1>(a, ncu, st, err) ||
                   run_resident<H, false, 0, 16, 2>(a, ncu, st, err) ||
                   run_resident<H, false, 0, 16, 3>(a, ncu, st, err) ||
                   run_resident<H, false, 0, 8, 10>(a, ncu, st, err);
        case 1:
            if (run_resident<H, false, 1, 16, 1>(a, ncu, st, err) ||
                run_resident<H, false, 1, 16, 2>(a, ncu, st, err))
                return true;
            if constexpr (H <= 3)
                return run_resident<H, false, 1, 16, 3>(a, ncu, st, err);
            else
                return run_resident<H, false, 1, 8, 6>(a, ncu, st, err);
        case 2:
            return run_resident<H, false, 2, 16, 1>(a, ncu, st, err) ||
                   run_resident<H, false, 2, 16, 2>(a, ncu, st, err) ||
                   run_resident<H, false, 2, 8, 6>(a, ncu, st, err);
        default: return false;
    }
}

}  // namespace

// stream null: only whether the grid is covered
bool launch_resident2d(Resident2D &a, int nd_case, int ncu, void *stream, int *err) {
    int e = 0;
    bool ok = false;
    SEIS_SWITCH_H(a.g.H, (ok = dispatch<HH>(a, nd_case, ncu, (hipStream_t)stream, e)));
    if (err) *err = e;
    return ok;
}

}  // namespace seis
