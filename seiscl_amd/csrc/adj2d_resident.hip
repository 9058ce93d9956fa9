// 2D adjoint runs resident on the chip: one launch makes the adjoint steps of a
// run.  fd2d_resident.hip describes the scheme; here a block also keeps the
// forward wavefields being backpropagated (L = 0) in LDS, or reads the forward
// state of every step from the recomputed history (L > 0), and holds its cells'
// gradient accumulators in registers.
//
// An adjoint step updates the stresses first: a block
//   1. adds the adjoint sources (and takes the last step's sources out of the
//      forward wavefields),
//   2. backpropagates the forward stresses (and puts the boundary shell back),
//      updates the adjoint ones and accumulates the M, mu and tau gradients:
//      its core and the rim of H cells (the gradients of the core only),
//   3. does the same with the velocities and the density gradient, core only,
//   4. applies the adjoint free surface of the next step to its core (it reads
//      the stresses of H columns on either side, which step 2 made),
//   5. publishes the velocities of its core's outer 2H cells and takes those
//      around its core.
// The first step's adjoint free surface is the caller's: nothing to do for
// wavefields of zero, the ordinary kernels otherwise.
//
// Values a step reads from memory (adjoint sources, boundary shell, history) are
// loaded as soon as the step before has used its own.
//
// Measured on MI355X, us per adjoint step, step kernels (elastic: replayed
// graphs) -> this kernel:
//                      100 x 100    200 x 400    300 x 800    433 x 1217
//   elastic FD4        15.6 -> 3.4  16.2 -> 4.4  19.9 -> 8.2  28.3 -> 15.0
//   elastic FD8        15.8 -> 4.9  17.1 -> 6.4  22.4 -> 10.3 not covered
//   + surface FD4      20.8 -> 4.5  22.3 -> 5.0  26.9 -> 10.0 36.5 -> 21.3
// and per step of a viscoelastic gradient (recomputation, checkpoints and adjoint;
// L = 2, FD4): 36 -> 13, 38 -> 17, 43 -> 20.  The exchange and the arithmetic of
// two runs bound it; a region's ten wavefields bound the grids that fit.
//
// Arithmetic: adjoint.hip, term by term.
#include "adj_terms.hpp"
#include "resident2d.hpp"

namespace seis {
namespace {

template <int H, int L, int NW, int N>
__global__ __launch_bounds__(64 * NW) void k_resident_adj2d(ResidentAdj2D a) {
    constexpr int RZ = 64 + 2 * H, RX = NW * N + 2 * H, FS = RX * RZ;
    constexpr bool BACK = L == 0;               // the forward run is run backwards
    constexpr int NF = BACK ? 10 : 5, NE = resident_adj_values(L);
    constexpr int NP = 8, NC = L ? 8 : 5, LS = L > 0 ? L : 1;
    constexpr int MR = (rim_cells(H, RX - 4 * H, RZ - 4 * H) + 64 * NW - 1) / (64 * NW);
    constexpr int NO = 6;                       // outputs of a receiver
    static_assert(RX * RZ <= 8192, "rlist packing");
    // fields 0-4: adjoint vx vz sxx szz sxz, 5-9: forward
    __shared__ float lds[NF * FS];
    __shared__ int rlist[kResidentMaxRec];
    __shared__ float xprof[6 * (kMaxNab + 1)];
    __shared__ float top[5][RX];                // free surface: M, mu, then hx, hz, ts
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
    const int rz0 = -H + bz * CZ - 2 * H, rx0 = -H + bx * CX - 2 * H;
    const int z = rz0 + H + lane, x0 = rx0 + H + w * N;
    const bool zpad = z >= -H && z < NZ + H, zin = z >= 0 && z < NZ;
    const bool core_z = lane >= H && lane < H + CZ, rim_z = lane < CZ + 2 * H;
    const bool edge_z = core_z && (lane < 3 * H || lane >= CZ - H);
    // the block whose core holds the surface row
    const bool surf = a.freesurf && -rz0 >= 2 * H && -rz0 < 2 * H + CZ;

    if (tid == 0) {
        rcount = 0;
        dead = 0;
        pulse = pulse_cell<H>(g, CZ, CX, rz0, rx0);
    }
    float *F = lds + (H + w * N) * RZ + H + lane;
    float co[NC][N], ps[NP][N], mv[3 * LS][N];
    // gradients of the core's cells, in registers (M, mu, rho) or, beside five
    // wavefields, in LDS (tau_p, tau_s too)
    constexpr int NG = BACK ? 3 : 5;
    __shared__ double lacc[BACK ? 1 : NG * NW * N * 64];
    double racc[BACK ? NG : 1][BACK ? N : 1];
    auto acc = [&](int q, int j) -> double & {
        if constexpr (BACK) return racc[q][j];
        else return lacc[(q * NW * N + w * N + j) * 64 + lane];
    };
    double *const ga[5] = {a.gM, a.gmu, a.grho, a.gtp, a.gts};
    float c1[N], c3[N], Ms[L ? N : 1], mus[L ? N : 1];
    int sm[BACK ? N : 1];                       // boundary-shell entry, -1: none
    const bool cpml = a.abs_type == 1;
    const bool zbot = z > NZ - NAB - 1;
    const bool pz = cpml && zin && (zbot || (!a.freesurf && z < NAB));
    const int kz = zbot ? z - NZ + 2 * NAB : z;
    // the lane's columns: in the grid and in the core or its rim; in the grid
    // and the core; in the core; in an x strip; among the core's outer 2H
    unsigned mrim = 0, mstr = 0, mcore = 0, mpx = 0, medge = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int c = w * N + j, x = x0 + j;
        const bool in = x >= 0 && x < NX, core = c >= H && c < H + CX;
        mrim |= (unsigned)(in && c < CX + 2 * H) << j;
        mstr |= (unsigned)(in && core) << j;
        mcore |= (unsigned)(core && x < NX + H) << j;
        medge |= (unsigned)(core && (c < 3 * H || c >= CX - H)) << j;
        mpx |= (unsigned)(cpml && in && (x < NAB || x > NX - NAB - 1)) << j;
    }
    mrim = __builtin_amdgcn_readfirstlane(mrim);
    mstr = __builtin_amdgcn_readfirstlane(mstr);
    mcore = __builtin_amdgcn_readfirstlane(mcore);
    medge = __builtin_amdgcn_readfirstlane(medge);
    mpx = __builtin_amdgcn_readfirstlane(mpx);
    Prof zp = {1, 0, 0, 1, 0, 0};
    for (int q = tid; q < FS; q += 64 * NW) {
        const int zz = rz0 + q % RZ, xx = rx0 + q / RZ;
        const bool in = zz >= -H && zz < NZ + H && xx >= -H && xx < NX + H;
        const long i = in ? g.idx(zz, 0, xx) : 0;
#pragma unroll
        for (int e = 0; e < 5; ++e) lds[e * FS + q] = in ? a.f[e][i] : 0.0f;
        if constexpr (BACK) {
#pragma unroll
            for (int e = 0; e < 5; ++e) lds[(5 + e) * FS + q] = in ? a.fw[e][i] : 0.0f;
        }
    }
    {
        const int zc = min(max(z, -H), NZ + H - 1);
        // cells outside the grid have no moduli: no gradient is kept there
        const int zg = min(max(z, 0), NZ - 1);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int x = x0 + j, xc = min(max(x, -H), NX + H - 1), xg = min(max(x, 0), NX - 1);
            const long i = g.idx(zc, 0, xc), ig = g.idx(zg, 0, xg);
#pragma unroll
            for (int q = 0; q < NC; ++q) co[q][j] = a.co[q][i];
#pragma unroll
            for (int q = 0; q < 3 * L; ++q) mv[q][j] = a.m[q / LS][(q % LS) * g.nfield + i];
#pragma unroll
            for (int q = 0; q < NP; ++q) ps[q][j] = 0;
#pragma unroll
            for (int q = 0; q < NG; ++q) acc(q, j) = ga[q][ig];
            float lM, lmu;
            if constexpr (L > 0) {
                lM = Ms[j] = a.Ms[ig];
                lmu = mus[j] = a.mus[ig];
            } else {
                lM = a.co[2][ig];
                lmu = a.co[3][ig];
            }
            c1[j] = mmu_c1_2d(lM, lmu);
            c3[j] = 1.0 / (lmu * lmu);
            if constexpr (BACK)
                sm[j] = zin && (mrim >> j & 1) ? (int)a.sh.inject(z + H, 0, x + H) : -1;
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
                    if ((q / 2) % 2 == 0) ps[q][j] = a.p[q][iz];
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
                    if ((q / 2) % 2 == 1) ps[q][j] = a.p[q][(long)ii * NZ + zi];
            }
        }
        if (cpml)
            for (int q = tid; q < 6 * (NAB + 1); q += 64 * NW)
                xprof[q] = a.cpml[(q % 6) * 2 * NAB + min(q / 6, 2 * NAB - 1)];
        if (surf)
            for (int q = tid; q < RX; q += 64 * NW) {
                const long i = g.idx(0, 0, min(max(rx0 + q, 0), NX - 1));
                top[0][q] = a.surfM[i];
                top[1][q] = a.surfmu[i];
            }
    }
    __syncthreads();
    // sources of the region, in order (L = 0: taken out of the forward run), and
    // the region's receivers
    int ns = 0;
    const float *ssrc = nullptr;
    float snext = 0;
    if constexpr (BACK) {
        int cell = -1, sz = 0, sx = 0;
        if (lane < a.s.nsrc) cell = a.s.src_cell[lane];
        bool here = cell >= 0 && !(a.freesurf && a.s.src_k[lane] < 2 * H);
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
                sfield[k] = source_field<false>(a.s.src_type[lane]);
                samp[k] = __int_as_float(lane);
            }
            __builtin_amdgcn_wave_barrier();
            if (lane < ns) {
                ssrc = a.s.src + (long)__float_as_int(samp[lane]) * a.NT;
                snext = ssrc[a.t1];
            }
        }
    }
    for (int r = tid; r < a.s.nrec; r += 64 * NW) {
        const int cell = a.s.rec_cell[r];
        if (cell < 0) continue;
        const int lx = cell / (int)g.ldz - g.H - rx0, lz = cell % (int)g.ldz - g.ZO - rz0;
        if (lx < 0 || lx >= CX + 4 * H || lz < 0 || lz >= CZ + 4 * H) continue;
        rlist[atomicAdd(&rcount, 1)] = r << 13 | (lx * RZ + lz);
    }
    int rl[MR], ri[MR];
#pragma unroll
    for (int e = 0; e < MR; ++e)
        rim_cell<H, RZ>(g, 0, CZ, CX, rz0, rx0, tid + e * 64 * NW, rl[e], ri[e]);
    __syncthreads();
    // (a block with more receivers than threads gives each thread several)
    constexpr int RT = (kResidentMaxRec + 64 * NW - 1) / (64 * NW);
    int myrec[RT];
    float rnext[RT][NO];
#pragma unroll
    for (int e = 0; e < RT; ++e)
        myrec[e] = tid + e * 64 * NW < rcount ? rlist[tid + e * 64 * NW] : -1;
    const bool recs = rcount > 0;
    auto res_load = [&](int t) {
#pragma unroll
        for (int e = 0; e < RT; ++e)
#pragma unroll
            for (int o = 0; o < NO; ++o)
                if (myrec[e] >= 0 && o < a.nout)
                    rnext[e][o] = a.res[((long)o * a.s.nrec + (myrec[e] >> 13)) * a.NT + t];
    };
    res_load(a.t1);
    const float *hc = a.hc;
    // shell or history of the next step's cells
    bool shell = false;
    float pre[5][N];
    if constexpr (BACK) {
#pragma unroll
        for (int j = 0; j < N; ++j) shell = shell || sm[j] >= 0;
    }
    const bool wave_shell = __any(shell);
    // (q0 .. q1 - 1 of vx vz sxx szz sxz)
    auto pre_load = [&](int t, int z, int x0, int q0, int q1) {
        if constexpr (BACK) {
            if (!wave_shell) return;
            const float *b = a.bnd + (long)(t - 1) * 5 * a.sh.n;
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (sm[j] >= 0) {
#pragma unroll
                    for (int q = 0; q < 5; ++q)
                        if (q >= q0 && q < q1) pre[q][j] = b[q * a.sh.n + sm[j]];
                }
        } else {
            if (!mstr || !core_z || !zin) return;
            const float *h = a.hist + (long)(t - a.hist_t0) * 5 * g.nfield;
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (mstr >> j & 1) {
                    const long i = g.idx(z, 0, x0 + j);
#pragma unroll
                    for (int q = 0; q < 5; ++q)
                        if (q >= q0 && q < q1) pre[q][j] = h[q * g.nfield + i];
                }
        }
    };
    pre_load(a.t1, z, x0, 0, 5);
    // sources of step t out of the forward run
    auto sources_out = [&](int t) {
        if constexpr (BACK) {
            if (ns && w == 0) {
                if (lane < ns) {
                    samp[lane] = snext;
                    if (t - 1 >= 0) snext = ssrc[t - 1];
                }
                __builtin_amdgcn_wave_barrier();
                if (lane == 0)
                    for (int q = 0; q < ns; ++q) {
                        const int c = scell[q], f = sfield[q];
                        const float amp = -1.0f * (a.DT * samp[q]);
                        if (f >= 0) lds[(5 + f) * FS + c] = lds[(5 + f) * FS + c] + amp;
                        else if (f == kSourceNormal)
                            for (int e = 7; e < 9; ++e)
                                lds[e * FS + c] =
                                    (float)((double)lds[e * FS + c] + (double)amp / 2.0);
                    }
            }
        }
    };

    const int x0_ = x0, z_ = z;
    for (int k = 0; k < a.nsteps; ++k) {
        const int t = a.t1 - k;
        // recomputed in every step: see fd2d_resident.hip
        int x0 = x0_, z = z_;
        asm volatile("" : "+s"(x0), "+v"(z));
        const unsigned tag = k + 1;
        Word *X = a.xch + (size_t)(tag & 1) * resident_nwords(NE) * g.nfield;
        const bool last = k + 1 == a.nsteps;
        // 1. adjoint sources (the forward run's were taken out after the exchange)
        if (recs) {
#pragma unroll
            for (int e = 0; e < RT; ++e) {
                if (myrec[e] < 0) continue;
                float *B = lds + (myrec[e] & 8191);
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    if (o >= a.nout) break;
                    const int code = a.code[o];
                    const float v = rnext[e][o];
                    if (code == O_P) {
                        const float q = v / 2.0f;
                        B[2 * FS] += q;
                        B[3 * FS] += q;
                    } else {
                        B[(code == O_VX    ? 0
                           : code == O_VZ  ? 1
                           : code == O_SXX ? 2
                           : code == O_SZZ ? 3
                                           : 4) * FS] += v;
                    }
                }
            }
            if (!last) res_load(t - 1);
            __syncthreads();
        }
        // 2. stresses of the core and its rim
        if (mrim) {
            float fa[N], fb[N], da[N], db[N];
            if constexpr (BACK) {
                dx<H, N, false, RZ>(F + 5 * FS, hc, fa);   // forward vxx
                dx<H, N, true, RZ>(F + 6 * FS, hc, fb);    // forward vzx
            }
            dx<H, N, false, RZ>(F, hc, da);
            dx<H, N, true, RZ>(F + FS, hc, db);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int x = x0 + j;
                if (!(mrim >> j & 1)) continue;
                float *f = F + j * RZ;
                float sxx, szz, sxz, gg, ff, d = 0, e = 0, fip, dip = 0;
                if constexpr (BACK) {
                    gg = co[2][j];
                    ff = 2.0 * co[3][j];
                    fip = co[4][j];
                    const float vxx = fa[j], vzx = fb[j];
                    const float vxz = dz<H, true>(f + 5 * FS, hc), vzz = dz<H, false>(f + 6 * FS, hc);
                    sxx = f[7 * FS];
                    szz = f[8 * FS];
                    sxz = f[9 * FS];
                    sxz -= (fip * (vxz + vzx));
                    sxx -= (gg * (vxx + vzz)) - (ff * vzz);
                    szz -= (gg * (vxx + vzz)) - (ff * vxx);
                    if (sm[j] >= 0) {
                        sxx = pre[2][j];
                        szz = pre[3][j];
                        sxz = pre[4][j];
                    }
                    if (zin && rim_z) {
                        f[7 * FS] = sxx;
                        f[8 * FS] = szz;
                        f[9 * FS] = sxz;
                    }
                } else {
                    gg = co[2][j];
                    ff = co[3][j];
                    d = co[4][j];
                    e = co[5][j];
                    fip = co[6][j];
                    dip = co[7][j];
                    sxx = pre[2][j];
                    szz = pre[3][j];
                    sxz = pre[4][j];
                }
                float vxx = da[j], vzx = db[j];
                float vxz = dz<H, true>(f, hc), vzz = dz<H, false>(f + FS, hc);
                const bool px = mpx >> j & 1;
                const int ii = x < NAB ? x : NX - x, ih = x < NAB ? x : NX - 1 - x;
                if (pz) {
                    pmlh(vxz, ps[4][j], zp);
                    pmlf(vzz, ps[5][j], zp);
                }
                if (px) {
                    const Prof xp = prof_x(xprof, ii, ih);
                    pmlf(vxx, ps[6][j], xp);
                    pmlh(vzx, ps[7][j], xp);
                }
                const bool keep = zin && core_z && (mstr >> j & 1);
                float lsxx, lszz, lsxz;
                if constexpr (BACK) {
                    lsxz = (fip * (vxz + vzx));
                    lsxx = (gg * (vxx + vzz)) - (ff * vzz);
                    lszz = (gg * (vxx + vzz)) - (ff * vxx);
                    if (zin && rim_z) {
                        f[2 * FS] = f[2 * FS] + lsxx;
                        f[3 * FS] = f[3 * FS] + lszz;
                        f[4 * FS] = f[4 * FS] + lsxz;
                    }
                } else {
                    const float DT2 = a.DT2;
                    float mxz = 0, mxx = 0, mzz = 0;
#pragma unroll
                    for (int l = 0; l < L; ++l) {
                        mxz += mv[2 * L + l][j];
                        mxx += mv[l][j];
                        mzz += mv[L + l][j];
                    }
                    lsxz = (fip * (vxz + vzx)) + (DT2 * mxz);
                    lsxx = ((gg * (vxx + vzz)) - (ff * vzz)) + (DT2 * mxx);
                    lszz = ((gg * (vxx + vzz)) - (ff * vxx)) + (DT2 * mzz);
                    const float oxz = mxz, oxx = mxx, ozz = mzz;
                    mxz = mxx = mzz = 0;
#pragma unroll
                    for (int l = 0; l < L; ++l) {
                        const float b = a.bl[l], c = a.cl[l], et = a.eta[l];
                        float &rxz = mv[2 * L + l][j], &rxx = mv[l][j], &rzz = mv[L + l][j];
                        rxz = b * (rxz * c - et * (dip * (vxz + vzx)));
                        rxx = b * (rxx * c - et * ((e * (vxx + vzz)) - (d * vzz)));
                        rzz = b * (rzz * c - et * ((e * (vxx + vzz)) - (d * vxx)));
                        mxz += rxz;
                        mxx += rxx;
                        mzz += rzz;
                    }
                    if (zin && rim_z) {
                        f[2 * FS] = f[2 * FS] + (lsxx + (DT2 * mxx));
                        f[3 * FS] = f[3 * FS] + (lszz + (DT2 * mzz));
                        f[4 * FS] = f[4 * FS] + (lsxz + (DT2 * mxz));
                    }
                    if (keep) {
                        const float vii[2] = {vxx, vzz};
                        const float Rm[2] = {DT2 * oxx + DT2 * mxx, DT2 * ozz + DT2 * mzz};
                        float Xp, Xs[2], tp, ts;
                        tau_parts_normal<float>(vxx + vzz, vii, Rm, 2, gg, ff, d, e, (float)L, a.DT,
                                                a.s0, Xp, Xs);
                        const float Xxz = tau_part_shear<float>(
                            vxz + vzx, DT2 * oxz + DT2 * mxz, fip, dip, lsxz + (DT2 * mxz),
                            (float)L, a.DT, a.s0);
                        const bool sh = tau_terms_2d(sxx, szz, sxz, Ms[j], mus[j], Xp, Xs[0], Xs[1],
                                                     Xxz, tp, ts);
                        acc(3, j) += (double)tp * a.gscale_s;
                        if (sh) acc(4, j) += (double)ts * a.gscale_s;
                    }
                }
                if (keep) {
                    const float c5 = 0.25 * c3[j];
                    const float dM = c1[j] * (sxx + szz) * (lsxx + lszz);
                    const float dmu = mmu_dmu_2d(dM, c3[j], c5, sxx, szz, sxz, lsxx, lszz, lsxz);
                    acc(1, j) += (double)dmu * a.gscale_s;
                    acc(0, j) += (double)-dM * a.gscale_s;
                }
            }
        }
        if (!last) pre_load(t - 1, z, x0, 2, 5);
        __syncthreads();
        // 3. velocities of the core
        if (mstr) {
            float fa[N], fb[N], da[N], db[N];
            if constexpr (BACK) {
                dx<H, N, true, RZ>(F + 7 * FS, hc, fa);    // forward sxx_x
                dx<H, N, false, RZ>(F + 9 * FS, hc, fb);   // forward sxz_x
            }
            dx<H, N, true, RZ>(F + 2 * FS, hc, da);
            dx<H, N, false, RZ>(F + 4 * FS, hc, db);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int x = x0 + j;
                if (!(mstr >> j & 1)) continue;
                float *f = F + j * RZ;
                const float rip = co[0][j], rkp = co[1][j];
                float vx, vz;
                if constexpr (BACK) {
                    const float szz_z = dz<H, true>(f + 8 * FS, hc);
                    const float sxz_z = dz<H, false>(f + 9 * FS, hc);
                    vx = f[5 * FS];
                    vz = f[6 * FS];
                    vx -= ((fa[j] + sxz_z) * rip);
                    vz -= ((szz_z + fb[j]) * rkp);
                    if (sm[j] >= 0) {
                        vx = pre[0][j];
                        vz = pre[1][j];
                    }
                } else {
                    vx = pre[0][j];
                    vz = pre[1][j];
                }
                float sxx_x = da[j], sxz_x = db[j];
                float szz_z = dz<H, true>(f + 3 * FS, hc), sxz_z = dz<H, false>(f + 4 * FS, hc);
                const bool px = mpx >> j & 1;
                const int ii = x < NAB ? x : NX - x, ih = x < NAB ? x : NX - 1 - x;
                if (pz) {
                    pmlf(sxz_z, ps[0][j], zp);
                    pmlh(szz_z, ps[1][j], zp);
                }
                if (px) {
                    const Prof xp = prof_x(xprof, ii, ih);
                    pmlh(sxx_x, ps[2][j], xp);
                    pmlf(sxz_x, ps[3][j], xp);
                }
                const float lvx = ((sxx_x + sxz_z) * rip);
                const float lvz = ((szz_z + sxz_x) * rkp);
                if (zin && core_z) {
                    float v[4] = {vx, f[0] + lvx, f[FS] + lvz, vz};
                    if constexpr (BACK) {
                        f[5 * FS] = vx;
                        f[6 * FS] = vz;
                    }
                    f[0] = v[1];
                    f[FS] = v[2];
                    const float d = -vx * lvx - vz * lvz;
                    if constexpr (BACK) acc(2, j) += d;
                    else acc(2, j) += (double)d * a.gscale_v;
                    if (!last && !surf && (edge_z || (medge >> j & 1))) {
                        const long i = g.idx(z, 0, x);
                        put_cell<NE>(X, g.nfield, i, BACK ? v : v + 1, tag);
                    }
                }
            }
        }
        if (!last) pre_load(t - 1, z, x0, 0, 2);
        // 4. adjoint free surface of the next step (k_surf_adj_a, k_surf_adj_b)
        if (surf && !last) {
            __syncthreads();
            const int row = -rz0;   // LDS row of z = 0
            for (int q = H + tid; q < 3 * H + CX; q += 64 * NW) {
                if (rx0 + q < 0 || rx0 + q >= NX) continue;
                const float lM = top[0][q], lmu = top[1][q];
                float *S = lds + q * RZ + row;
                float lsxx = S[2 * FS], lszz = S[3 * FS];
                const float temp1 = lsxx, temp2 = lszz;
                const float aa = 1.0f / (4.0f * lM * lmu - 4.0f * lmu * lmu);
                lsxx = -aa * (lM * temp1 + (-lM + 2.0f * lmu) * temp2);
                lszz = -aa * (lM * temp2 + (-lM + 2.0f * lmu) * temp1);
                lszz = 0.0;
                top[2][q] = -((lM - lmu * 2.0f) * (lM - lmu * 2.0f) / lM);
                top[3][q] = -(lM - lmu * 2.0f);
                top[4][q] = lsxx;
                S[3 * FS] = -(lM * lszz + (lM - 2.0f * lmu) * lsxx);
                S[2 * FS] = -(lM * lsxx + (lM - 2.0f * lmu) * lszz);
            }
            __syncthreads();
            if (mstr && z >= 0 && z < H && core_z) {
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    if (!(mstr >> j & 1)) continue;
                    const int x = x0 + j, q = H + w * N + j;
                    float *f = F + j * RZ;
                    if (z == 0) {
                        float v = f[0];
                        const float rip = co[0][j];
#pragma unroll
                        for (int s = -(H - 1); s <= H; ++s) {
                            const int xs = x + s;
                            if (xs < 0 || xs >= NX) continue;
                            const int c = q + s;
                            if (s <= 0) v += (hc[1 - s] * top[2][c] * top[4][c] * rip);
                            else v += (-hc[s] * top[2][c] * top[4][c] * rip);
                        }
                        f[0] = v;
                    }
                    // hc[1 + z] as a constant index: z differs from lane to lane
                    float h = hc[1];
#pragma unroll
                    for (int m = 1; m < H; ++m) h = z == m ? hc[1 + m] : h;
                    f[FS] += (h * top[3][q] * top[4][q] * co[1][j]);
                }
            }
            __syncthreads();
            if (mstr && zin && core_z) {
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    if (!(mstr >> j & 1) || !(edge_z || (medge >> j & 1))) continue;
                    const float *f = F + j * RZ;
                    const float v[4] = {BACK ? f[5 % NF * FS] : 0.0f, f[0], f[FS],
                                        BACK ? f[6 % NF * FS] : 0.0f};
                    put_cell<NE>(X, g.nfield, g.idx(z, 0, x0 + j), BACK ? v : v + 1, tag);
                }
            }
        }
        // 5. the rim's velocities
        if (last) break;
        const bool ok = take_rim<NE, MR>(X, g.nfield, tag, a.patience, ri, [&](int e, const float *u) {
            if constexpr (BACK) {
                lds[5 * FS + rl[e]] = u[0];
                lds[rl[e]] = u[1];
                lds[FS + rl[e]] = u[2];
                lds[6 * FS + rl[e]] = u[3];
            } else {
                lds[rl[e]] = u[0];
                lds[FS + rl[e]] = u[1];
            }
        });
        if (!ok && lane == 0) dead = 1;
        __syncthreads();
        if (dead) break;
        if (BACK && ns) {
            sources_out(t);
            __syncthreads();
        }
    }
    if constexpr (BACK) {
        __syncthreads();
        sources_out(a.t1 - a.nsteps + 1);
    }
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
        for (int q = 0; q < 5; ++q) a.f[q][i] = F[q * FS + j * RZ];
        if constexpr (BACK) {
#pragma unroll
            for (int q = 0; q < 5; ++q) a.fw[q][i] = F[(5 + q) * FS + j * RZ];
        }
        if (!zin || x < 0 || x >= NX) continue;
#pragma unroll
        for (int q = 0; q < 3 * L; ++q) a.m[q / LS][(q % LS) * g.nfield + i] = mv[q][j];
#pragma unroll
        for (int q = 0; q < NG; ++q) ga[q][i] = acc(q, j);
        const bool px = mpx >> j & 1;
        const int ii = x < NAB ? x : x - NX + 2 * NAB;
        const long iz = (long)x * 2 * NAB + kz, ix = (long)ii * NZ + z;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const bool isz = (q / 2) % 2 == 0;
            if (isz ? pz : px) a.p[q][isz ? iz : ix] = ps[q][j];
        }
    }
}

template <int H, int L, int NW, int N>
bool run_adj(ResidentAdj2D &a, int ncu, hipStream_t st, int &err) {
    const Tiling t = tiling(a.g, NW * N, ncu);
    if (!t.nbz) return false;
    a.cz = t.cz;
    a.cx = t.cx;
    a.nbz = t.nbz;
    a.ntile = (unsigned)(t.nbz * t.nbx);
    if (!st) return true;
    hipLaunchKernelGGL((k_resident_adj2d<H, L, NW, N>), dim3((a.ntile + 7) / 8 * 8), dim3(64, NW), 0, st, a);
    err = (int)hipGetLastError();
    return true;
}

// The smallest region that covers the grid; ten wavefields of 48 columns fit
// the LDS up to FD order 6.
template <int H>
bool dispatch_adj(ResidentAdj2D &a, int L, int ncu, hipStream_t st, int &err) {
    switch (L) {
        case 0:
            if (run_adj<H, 0, 16, 1>(a, ncu, st, err) || run_adj<H, 0, 8, 4>(a, ncu, st, err))
                return true;
            if constexpr (H <= 3) return run_adj<H, 0, 8, 6>(a, ncu, st, err);
            else return false;
        case 1:
            return run_adj<H, 1, 16, 1>(a, ncu, st, err) || run_adj<H, 1, 8, 4>(a, ncu, st, err);
        case 2:
            return run_adj<H, 2, 16, 1>(a, ncu, st, err) || run_adj<H, 2, 8, 4>(a, ncu, st, err);
        default: return false;
    }
}

}  // namespace

// stream null: only whether the grid is covered
bool launch_resident_adj2d(ResidentAdj2D &a, int L, int ncu, void *stream, int *err) {
    int e = 0;
    bool ok = false;
    SEIS_SWITCH_H(a.g.H, (ok = dispatch_adj<HH>(a, L, ncu, (hipStream_t)stream, e)));
    if (err) *err = e;
    return ok;
}

}  // namespace seis
