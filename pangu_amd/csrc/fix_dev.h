// Device code of FixPrimitive and the conserved state of one cell.
#pragma once
#include <hip/hip_runtime.h>

#include "cell_dev.h"
#include "common.h"
#include "kernels.h"
#include "physics_dev.h"

namespace pangu {

// ------------------------------------------------ fix_primitive + conservative
// FixPrimitive over the entire block (primitive_fixer.cc:64-166) and, for
// interior cells, CalculateConservative (conservative.cc:57-107).  The
// primitives and conservatives are written with non-temporal stores: on
// MI355X that leaves L2 to the stencil reads of the flux sweep that follows
// (measured 1 % faster per cycle on the 3-D torus than ordinary stores).
// One cell of k_fix_cons.  write = false computes without storing (a halo
// cell of k_fix_flux_x1, which another workgroup owns); pout (optional)
// receives the fixed primitives, every slot.
template <int MF, bool FIX, bool CONS, bool HB, bool HK>
__device__ __forceinline__ void fix_cons_cell(const KCtx &C, const KFields &F, uint8_t *const *mask, int b,
                                              int k, int j, int i, bool write, double *pout) {
  const DevBlock &B = C.blk[b];
  const bool interior = i >= B.s[0] && i <= B.e[0] && j >= B.s[1] && j <= B.e[1] &&
                        k >= B.s[2] && k <= B.e[2];
  if (!FIX && !interior) return;
  const DevGeo &G = C.geo[B.geo];
  const int64_t t = cen_index(G, k, j, i);
  const int64_t id = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  constexpr int NC = ncomp<HB, HK>();
  gptr<double> pp[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) pp[q] = glb(F.prim[b * NC + q]);
  double p[NPRIM];
#pragma unroll
  for (int s = 0; s < NPRIM; ++s) p[s] = 0.0;
#pragma unroll
  for (int q = 0; q < NC; ++q) p[slot_of<HB, HK>(q)] = pp[q][id];
  CenLoad m;
  load_cen_state<MF>(G, t, m);
  const Phys &P = C.ph;
  if (FIX) {
    const double small = 1.0e-20;
    const double sms = kmax(P.sigma_max, small);
    const double rho_before = kmax(p[RHO], small);
    double rho_floor = ldc32(G.cen, (int64_t)CG_RHOFL * G.ncen, (uint32_t)t);
    const double eng_floor = ldc32(G.cen, (int64_t)CG_ENGFL * G.ncen, (uint32_t)t);
    St st;
    calc_state<MF, HB>(p, m.g, m.gc0, m.alpha, st);
    const double rho = p[RHO], ug = p[ENY];
    uint8_t mk = 0;
    if (rho_floor < ug / sms) rho_floor = ug / sms;
    const double sigma = st.bsq / rho;
    if (sigma > P.sigma_max) {
      rho_floor = st.bsq / sms;
      mk |= 8;
    }
    if (p[RHO] < rho_floor) {
      p[RHO] = rho_floor;
      mk |= 1;
    }
    if (p[ENY] < eng_floor) {
      p[ENY] = eng_floor;
      mk |= 2;
    }
    const double u1 = p[UX1], u2 = p[UX2], u3 = p[UX3];
    const double *g = m.g;
    double uvsq = g[5] * u1 * u1 + g[10] * u2 * u2 + g[15] * u3 * u3;
    if (g_dense<MF>()) uvsq = uvsq + 2.0 * (g[6] * u1 * u2 + g[7] * u1 * u3 + g[11] * u2 * u3);
    if (MF == FORM_POLOIDAL) uvsq = uvsq + 2.0 * (g[7] * u1 * u3);
    const double umax2 = P.lorentz_max * P.lorentz_max - 1.0;
    if (umax2 > 0.0 && uvsq > umax2) {
      const double f = sqrt(umax2 / kmax(uvsq, small));
      p[UX1] *= f;
      p[UX2] *= f;
      p[UX3] *= f;
      mk |= 4;
    }
    const double rho_after = kmax(p[RHO], small);
    if (HK && rho_after != rho_before) p[KEL] *= pow(rho_after / rho_before, -P.gamma);
    p[ENT] = (P.gamma - 1.0) * p[ENY] * pow(p[RHO], -P.gamma);
    if (HK) p[KEL] = clamp_by_ratio(P.ratio_min, P.ratio_max, p[ENT], p[KEL]);
    if (P.metric == PANGU_METRIC_CKS && ldc32(G.cen, (int64_t)CG_RAD * G.ncen, (uint32_t)t) < P.r_excise) {
      const double e_exc = P.pexcise / (P.gamma - 1.0);
      p[RHO] = P.dexcise;
      p[ENY] = e_exc;
      p[UX1] = 0.0;
      p[UX2] = 0.0;
      p[UX3] = 0.0;
      p[ENT] = (P.gamma - 1.0) * e_exc * pow(P.dexcise, -P.gamma);
      if (HK) p[KEL] = e_exc;
      mk |= 16;
    }
    // rho, u and u~ change only where a floor, the Lorentz cap or excision
    // set a mask bit; elsewhere memory already holds them (the entropy is
    // recomputed in every cell)
    if (write && mk) {
      __builtin_nontemporal_store(p[RHO], &pp[0][id]);
      __builtin_nontemporal_store(p[ENY], &pp[1][id]);
      __builtin_nontemporal_store(p[UX1], &pp[2][id]);
      __builtin_nontemporal_store(p[UX2], &pp[3][id]);
      __builtin_nontemporal_store(p[UX3], &pp[4][id]);
    }
    if (write) {
      __builtin_nontemporal_store(p[ENT], &pp[ient<HB>()][id]);
      if (HK) pp[ikel<HB>()][id] = p[KEL];
      if (mask) glb(mask[b])[id] = mk;
    }
  }
  if (pout) {
#pragma unroll
    for (int q = 0; q < NPRIM; ++q) pout[q] = p[q];
  }
  if (CONS && interior && write) {
    St st;
    calc_state<MF, HB>(p, m.g, m.gc0, m.alpha, st);
    double f[NPRIM];
    contravariant_flux<0, HB>(P.gamma, p, st, m.sg, f);
#pragma unroll
    for (int q = 0; q < NC; ++q) __builtin_nontemporal_store(f[slot_of<HB, HK>(q)], &glb(F.cons[b * NC + q])[id]);
  }
}

}  // namespace pangu
