// Gradient increments of one cell and step, shared by the adjoint step kernels
// and the resident adjoint runs.
#pragma once
#include <hip/hip_runtime.h>

namespace seis {
namespace {

// M and mu in 2D (src/update_adjs2D.cl:441-456): dM = c1 (sum s)(sum ls), and
// mu's increment from it.
template <typename R>
__device__ __forceinline__ R mmu_c1_2d(R lM, R lmu) {
    return 1.0 / ((2.0 * lM - 2.0 * lmu) * (2.0 * lM - 2.0 * lmu));
}
template <typename R>
__device__ __forceinline__ R mmu_dmu_2d(R dM, R c3, R c5, R sxx, R szz, R sxz, R lsxx, R lszz,
                                        R lsxz) {
    return -c3 * (sxz * lsxz) + dM - c5 * ((sxx - szz) * (lsxx - lszz));
}

// tau gradients of the GSLS stress update (no counterpart in the
// reference's time-domain kernels, which declare gradtaup/gradtaus and never
// write them, src/update_adjs3D.cl:66; its DFT path forms them in
// src/calc_grad.c:111-152).  A normal-stress update is
//   inc_ii = g th - f (th - v_ii) + Rm_ii,  g = M(1+L tp), f = 2mu(1+L ts),
// Rm_ii = DT2 sum_l (r_ii,l old + new): the whole memory term of the step,
// the memory variables forced by e th - d (th - v_ii), e = M tp/DT,
// d = 2 mu ts/DT, through the same relaxation filters, so Rm_ii = e F -
// d F_ii and sum_ii Rm_ii = (ND e - (ND-1) d) F.  The change of the update
// with tp (at fixed M) is M L th + (M/DT) F, with ts (at fixed mu)
// -2mu L (th - v_ii) - (e F - Rm_ii)/ts, and for a shear component (pair
// mu_ij(1+L ts_ij), mu_ij ts_ij/DT) mu_ij L w_ij + Rm_ij/ts_ij.  Holding the
// wave speeds through the normalisation M = M_f0/(1 + s0 tp) adds
// -s0/(1+s0 tp) times the part linear in M (likewise for mu).  M, mu, tp, ts
// are recovered from g, f, d, e.  Cells with ts = 0 drop the memory term of
// ts.  The gradient is minus the forward strain (the forward stresses
// through the compliance of the gradient moduli, as for M and mu) times
// these changes.
template <typename R>
__device__ __forceinline__ void tau_parts_normal(R theta, const R *vii, const R *Rm, int nd, R g,
                                                 R f, R d, R e, R L, R DT, R s0, R &Xp, R *Xs) {
    const R MR = g - L * e * DT;
    const R tp = e * DT / MR;
    const R tmu = f - L * d * DT;
    const R ts = tmu != R(0) ? d * DT / tmu : R(0);
    const R kp = s0 / (R(1) + s0 * tp);
    const R ks = s0 / (R(1) + s0 * ts);
    const R den = nd == 3 ? R(3) * e - R(2) * d : R(2) * e - d;
    const R trm = nd == 3 ? (Rm[0] + Rm[1]) + Rm[2] : Rm[0] + Rm[1];
    const R F = den != R(0) ? trm / den : R(0);
    Xp = (MR * L - kp * g) * theta + (MR / DT - kp * e) * F;
    for (int k = 0; k < nd; ++k) {
        const R dev = theta - vii[k];
        const R q = e * F - Rm[k];
        const R Sk = -(f * dev) - q;
        Xs[k] = -(tmu * L * dev) - (ts > R(0) ? q / ts : R(0)) - ks * Sk;
    }
}

template <typename R>
__device__ __forceinline__ R tau_part_shear(R w, R Rm, R fij, R dij, R inc, R L, R DT, R s0) {
    const R mua = fij - L * dij * DT;
    const R tsa = mua != R(0) ? dij * DT / mua : R(0);
    const R ksa = s0 / (R(1) + s0 * tsa);
    return mua * L * w + (tsa > R(0) ? Rm / tsa : R(0)) - ksa * inc;
}

// tau_p's and tau_s's increments in 2D; false: mu = 0, no tau_s term
template <typename R>
__device__ __forceinline__ bool tau_terms_2d(R sxx, R szz, R sxz, R lM, R lmu, R Xp, R Xxx, R Xzz,
                                             R Xxz, R &tp, R &ts) {
    const R lam = lM - R(2) * lmu;
    const R th = (sxx + szz) / (R(2) * lM - R(2) * lmu);
    tp = -(th * Xp);
    ts = 0;
    if (lmu == R(0)) return false;
    const R exx = (sxx - lam * th) / (R(2) * lmu);
    const R ezz = (szz - lam * th) / (R(2) * lmu);
    const R gxz = sxz / lmu;
    ts = -((exx * Xxx + ezz * Xzz) + gxz * Xxz);
    return true;
}

}  // namespace
}  // namespace seis
