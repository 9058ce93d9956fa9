// Results on their way to the caller: gradients taken to the parameterisation
// and seismograms brought into the caller's layout on the GPU, and copies of
// many arrays in one launch.
//
// On the host the gradient transform (src/calc_grad.c:975-1110) took three
// accumulators in double over PCIe, two passes of strided loops and one division
// and square root per cell and parameter on one thread: 44 ms for 2.1 million
// cells, and 20 ms more to transpose the result.  Here a kernel bound by the
// 36 bytes it reads and 12 it writes per cell does both.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "seis_internal.hpp"

namespace seis {
namespace {

constexpr int TT = 32;   // transposed tile

// transf_grad (grad_host.cpp) of one cell, in double
__device__ __forceinline__ void transform_cell(const GradOut &a, long i, double lM, double lmu,
                                               float *out) {
    const double dt = a.dt, dh = a.dh;
    const double rho = 1.0 / a.rho[i] * dt / dh;
    const double M = lM * dh / dt, mu = lmu * dh / dt;
    double gr = a.g[2][i] / dt, gm = a.g[0][i] / dt, gu = a.g[1][i] / dt;
    if (a.rho_fix) gr *= dh * dh / (dt * dt);
    if (a.param_type == 0 || a.param_type == 2) {
        gr = gr + M / rho * gm;
        if (mu > 0) gr = gr + mu / rho * gu;
        if (a.param_type == 0) {
            gm = 2.0 * sqrt(rho * M) * gm;
            gu = 2.0 * sqrt(rho * mu) * gu;
        } else {
            gm = 2.0 * sqrt(M / rho) * gm;
            gu = 2.0 * sqrt(mu / rho) * gu;
        }
    }
    out[0] = (float)gm;
    out[1] = (float)gu;
    out[2] = (float)gr;
}

// One block: 32 z x 32 x of one y.  The accumulators are read along z; with
// a.model the result is turned in LDS and written along x ([NZ][NY][NX]), else
// along z ([NX][NY][NZ]).
template <typename R>
__global__ __launch_bounds__(TT * 8) void k_grad_out(GradOut a) {
    __shared__ float t[5][TT][TT + 1];
    const Layout &g = a.lay;
    const int z0 = blockIdx.x * TT, x0 = blockIdx.y * TT, y = blockIdx.z;
    const long n = (long)g.NZ * g.NY * g.NX;
    for (int r = threadIdx.y; r < TT; r += 8) {
        const int z = z0 + threadIdx.x, x = x0 + r;
        if (z >= g.NZ || x >= g.NX) continue;
        const long i = g.idx(z, y, x);
        float v[5] = {0, 0, 0, 0, 0};
        if (a.out)
            transform_cell(a, i, (double)((const R *)a.Ms)[i], (double)((const R *)a.mus)[i], v);
        if (a.tau) {
            v[3] = (float)(a.g[3][i] * a.ktau);
            v[4] = (float)(a.g[4][i] * a.ktau);
        }
        if (a.model) {
#pragma unroll
            for (int q = 0; q < 5; ++q) t[q][r][threadIdx.x] = v[q];
        } else {
            const long o = ((long)x * g.NY + y) * g.NZ + z;
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                if (q < 3 && a.out) a.out[q * n + o] = v[q];
                if (q >= 3 && a.tau) a.tau[(q - 3) * n + o] = v[q];
            }
        }
    }
    if (!a.model) return;
    __syncthreads();
    for (int r = threadIdx.y; r < TT; r += 8) {
        const int z = z0 + r, x = x0 + threadIdx.x;
        if (z >= g.NZ || x >= g.NX) continue;
        const long o = ((long)z * g.NY + y) * g.NX + x;
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            if (q < 3 && a.out) a.out[q * n + o] = t[q][threadIdx.x][r];
            if (q >= 3 && a.tau) a.tau[(q - 3) * n + o] = t[q][threadIdx.x][r];
        }
    }
}

// [NT][nout][nrec] -> [nout][NT][nrec]
template <typename T>
__global__ void k_seis_rows(const T *in, float *out, int NT, int nout, int nrec) {
    const long n = (long)NT * nout * nrec;
    for (long k = blockIdx.x * (long)blockDim.x + threadIdx.x; k < n;
         k += (long)gridDim.x * blockDim.x) {
        const long r = k % nrec, o = (k / nrec) % nout, t = k / ((long)nrec * nout);
        out[(o * NT + t) * nrec + r] = (float)in[k];
    }
}

// Every array of the list, 16 bytes per lane where both ends allow it.
__global__ void k_copy_list(CopyList c) {
    const int q = blockIdx.y;
    const char *src = (const char *)c.src[q];
    char *dst = (char *)c.dst[q];
    const size_t n = c.bytes[q];
    const size_t step = (size_t)gridDim.x * blockDim.x;
    size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((((size_t)src | (size_t)dst | n) & 15) == 0) {
        for (; k < n / 16; k += step) ((uint4 *)dst)[k] = ((const uint4 *)src)[k];
    } else if ((((size_t)src | (size_t)dst | n) & 3) == 0) {
        for (; k < n / 4; k += step) ((uint32_t *)dst)[k] = ((const uint32_t *)src)[k];
    } else {
        for (; k < n; k += step) dst[k] = src[k];
    }
}

}  // namespace

void launch_grad_out(const GradOut &a, bool f64, void *stream) {
    const Layout &g = a.lay;
    const dim3 grid((g.NZ + TT - 1) / TT, (g.NX + TT - 1) / TT, g.NY), blk(TT, 8);
    if (f64) hipLaunchKernelGGL(k_grad_out<double>, grid, blk, 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(k_grad_out<float>, grid, blk, 0, (hipStream_t)stream, a);
}

void launch_seis_rows(const void *in, bool f64, float *out, int NT, int nout, int nrec,
                      void *stream) {
    const long n = (long)NT * nout * nrec;
    if (n <= 0) return;
    const int blocks = (int)std::min<long>((n + 255) / 256, 4096);
    if (f64)
        hipLaunchKernelGGL(k_seis_rows<double>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const double *)in, out, NT, nout, nrec);
    else
        hipLaunchKernelGGL(k_seis_rows<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const float *)in, out, NT, nout, nrec);
}

void launch_copy_list(const CopyList &c, void *stream) {
    if (c.n <= 0) return;
    size_t most = 0;
    for (int q = 0; q < c.n; ++q) most = std::max(most, c.bytes[q]);
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>((most + 4095) / 4096, 2048));
    hipLaunchKernelGGL(k_copy_list, dim3(blocks, c.n), dim3(256), 0, (hipStream_t)stream, c);
}

}  // namespace seis
