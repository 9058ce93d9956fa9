// What the resident 2D kernels share: stencils on LDS tiles, CPML, the exchange
// of rim cells between blocks, the agreement at the end of a run.
// fd2d_resident.hip describes the scheme.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fd_common.hpp"
#include "resident_tiles.hpp"
#include "seis_internal.hpp"

namespace seis {
namespace {

// x-derivatives of N consecutive cells; f: the lane's first cell in LDS.
// PLUS: forward (Dp), else backward (Dm), with their terms and order.
template <int H, int N, bool PLUS, int RZ>
__device__ __forceinline__ void dx(const float *f, const float *hc, float *d) {
    constexpr int W = N + 2 * H - 1, O = PLUS ? H - 1 : H;
    float w[W];
#pragma unroll
    for (int k = 0; k < W; ++k) w[k] = f[(k - O) * RZ];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        float acc = PLUS ? hc[1] * (w[j + O + 1] - w[j + O]) : hc[1] * (w[j + O] - w[j + O - 1]);
#pragma unroll
        for (int k = 2; k <= H; ++k)
            acc = acc + (PLUS ? hc[k] * (w[j + O + k] - w[j + O - k + 1])
                              : hc[k] * (w[j + O + k - 1] - w[j + O - k]));
        d[j] = acc;
    }
}
template <int H, bool PLUS>
__device__ __forceinline__ float dz(const float *f, const float *hc) {
    float acc = PLUS ? hc[1] * (f[1] - f[0]) : hc[1] * (f[0] - f[-1]);
#pragma unroll
    for (int k = 2; k <= H; ++k)
        acc = acc + (PLUS ? hc[k] * (f[k] - f[1 - k]) : hc[k] * (f[k - 1] - f[-k]));
    return acc;
}

struct Prof {       // CPML profile at one cell: K, a, b on the full and half grid
    float K, a, b, Kh, ah, bh;
};
__device__ __forceinline__ Prof prof_load(const float *c, int n, int kf, int kh) {
    return {c[CK * n + kf], c[CA * n + kf], c[CB * n + kf],
            c[CKH * n + kh], c[CAH * n + kh], c[CBH * n + kh]};
}
// the same from the block's LDS copy, six values per profile index
__device__ __forceinline__ Prof prof_x(const float *p, int kf, int kh) {
    return {p[6 * kf + CK], p[6 * kf + CA], p[6 * kf + CB],
            p[6 * kh + CKH], p[6 * kh + CAH], p[6 * kh + CBH]};
}
__device__ __forceinline__ void pmlf(float &d, float &psi, const Prof &p) {
    psi = p.b * psi + p.a * d;
    d = d / p.K + psi;
}
__device__ __forceinline__ void pmlh(float &d, float &psi, const Prof &p) {
    psi = p.bh * psi + p.ah * d;
    d = d / p.Kh + psi;
}

// The field a source of a type feeds: 0 vx, 1 vz, 2 p, the normal stresses, or none.
// A y force has no vy to feed and goes to the normal stresses, as in the step
// kernels (sources_body).
constexpr int kSourceNormal = -1, kSourceNone = -2;
template <bool ACOUSTIC>
__device__ __forceinline__ int source_field(int type) {
    if (type == 0) return 0;
    if (type == 2) return 1;
    if (type == 3 || type == 100) return ACOUSTIC ? 2 : kSourceNormal;
    return type == 1 && !ACOUSTIC ? kSourceNormal : kSourceNone;
}

using Word = unsigned long long;
__device__ __forceinline__ void put_word(Word *p, Word v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ Word get_word(const Word *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The words of one cell: NE exchanged values (1, 2, 3 or 4) and the number of
// their step (tag > 0), 32 bits of it beside one value, 16 bits otherwise.
template <int NE>
__device__ __forceinline__ void put_cell(Word *X, long plane, long i, const float *v, unsigned tag) {
    if constexpr (NE <= 2) {
#pragma unroll
        for (int q = 0; q < NE; ++q)
            put_word(X + q * plane + i, (Word)tag << 32 | __float_as_uint(v[q]));
    } else {
        // the halves of one value ride beside the others
        const unsigned m = __float_as_uint(v[1]), t = tag << 16;
        put_word(X + i, (Word)(t | m >> 16) << 32 | __float_as_uint(v[0]));
        put_word(X + plane + i, (Word)(t | (m & 0xffff)) << 32 | __float_as_uint(v[2]));
        if constexpr (NE == 4) put_word(X + 2 * plane + i, (Word)t << 32 | __float_as_uint(v[3]));
    }
}
template <int NE>
__device__ __forceinline__ void get_cell(const Word *X, long plane, long i, Word *w) {
#pragma unroll
    for (int q = 0; q < resident_nwords(NE); ++q) w[q] = get_word(X + q * plane + i);
}
template <int NE>
__device__ __forceinline__ bool cell_ready(const Word *w, unsigned tag) {
    bool r = true;
#pragma unroll
    for (int q = 0; q < resident_nwords(NE); ++q)
        r = r && (NE <= 2 ? (unsigned)(w[q] >> 32) == tag : (unsigned)(w[q] >> 48) == (tag & 0xffff));
    return r;
}
template <int NE>
__device__ __forceinline__ void cell_values(const Word *w, float *v) {
    if constexpr (NE <= 2) {
#pragma unroll
        for (int q = 0; q < NE; ++q) v[q] = __uint_as_float((unsigned)w[q]);
    } else {
        v[0] = __uint_as_float((unsigned)w[0]);
        v[1] = __uint_as_float((unsigned)(w[0] >> 32) << 16 | ((unsigned)(w[1] >> 32) & 0xffff));
        v[2] = __uint_as_float((unsigned)w[1]);
        if constexpr (NE == 4) v[3] = __uint_as_float((unsigned)w[2]);
    }
}

// Waits for the words of a thread's rim cells and hands their values to
// put(e, values); false if that took longer than patience.  The first cell is
// waited for alone and the others are loaded once it is there (they are then, as
// a rule, too): polling all of them in vain keeps the memory path busy.
template <int NE, int MR, typename F>
__device__ __forceinline__ bool take_rim(const Word *X, long plane, unsigned tag,
                                         long long patience, const int *ri, F &&put) {
    Word v[MR][resident_nwords(NE)];
    const long long start = wall_clock64();
    auto take = [&](auto first, auto end) {
        constexpr int E0 = decltype(first)::value, E1 = decltype(end)::value;
        while (true) {
            bool wait = false;
#pragma unroll
            for (int e = E0; e < E1; ++e)
                if (ri[e] >= 0) get_cell<NE>(X, plane, ri[e], v[e]);
#pragma unroll
            for (int e = E0; e < E1; ++e)
                if (ri[e] >= 0 && !cell_ready<NE>(v[e], tag)) wait = true;
            if (!__any(wait)) break;
            if (wall_clock64() - start > patience) return false;
        }
        return true;
    };
    if (!take(std::integral_constant<int, 0>(), std::integral_constant<int, 1>())) return false;
    if constexpr (MR > 1)
        if (!take(std::integral_constant<int, 1>(), std::integral_constant<int, MR>())) return false;
#pragma unroll
    for (int e = 0; e < MR; ++e)
        if (ri[e] >= 0) {
            float u[NE];
            cell_values<NE>(v[e], u);
            put(e, u);
        }
    return true;
}

// One thread per block, when its block has made its last step (or given up):
// 1 once every block of the run has made its last step, 2 if the run failed.
// sync[0] counts blocks, sync[1] is the run's state, which the last block or one
// that gave up sets, whichever is first.  A block of halo cells is here as soon as
// it has recorded its receivers: it goes on waiting while a neighbour makes steps
// (pulse: a word of the neighbour's, null for other blocks).
__device__ __forceinline__ int agree(int *sync, int *failed, int nblocks, int gave_up,
                                     long long patience, const Word *pulse) {
    int st = gave_up ? 2 : 0;
    if (!gave_up) {
        if (__hip_atomic_fetch_add(sync, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 == nblocks)
            st = 1;
        long long start = wall_clock64();
        Word seen = pulse ? get_word(pulse) : 0;
        while (!st) {
            // (acquired by the exchange below)
            st = __hip_atomic_load(sync + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (st) break;
            if (wall_clock64() - start > patience) {
                const Word now = pulse ? get_word(pulse) : seen;
                if (now == seen) st = 2;
                seen = now;
                start = wall_clock64();
            }
            __builtin_amdgcn_s_sleep(4);
        }
    }
    int open = 0;
    if (!__hip_atomic_compare_exchange_strong(sync + 1, &open, st, __ATOMIC_ACQ_REL,
                                              __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT))
        st = open;
    if (st == 2) __hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return st;
}

}  // namespace
}  // namespace seis
