// Device code of the flux sweeps: reconstruction, face physics and the
// Riemann combine of one face.
#pragma once
#include <hip/hip_runtime.h>

#include "cell_dev.h"
#include "common.h"
#include "kernels.h"
#include "physics_dev.h"

namespace pangu {

// ------------------------------------------------------------- flux sweep
// One direction of CalculateLAXF / CalculateHLL (laxf.cc:78-181 and the
// X2/X3 twins): reconstruction of every primitive, face metric, fast speeds,
// four contravariant fluxes and the Riemann combine.  Face (k,j,i) is the
// lower face of cell (k,j,i) along DIR.
// Face physics of one sweep direction for face (k, j, i) of block b, the
// lower face of cell (k, j, i) along DIR: face metric, fluid states, fast
// speeds, the four contravariant fluxes and the Riemann combine, from the
// reconstructed left (pl) and right (pr) primitives.
template <int DIR, int RS, bool HB, bool HK, int MF>
__device__ __forceinline__ void face_flux(const KCtx &C, const KFields &F, double *const *alfven, int b,
                                          int k, int j, int i, const double pl[NPRIM],
                                          const double pr[NPRIM]) {
  const DevBlock &B = C.blk[b];
  const int64_t id = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  constexpr int NC = ncomp<HB, HK>();
  const DevGeo &G = C.geo[B.geo];
  double g[16], gc0[4], gdd = 1.0, sg = 1.0, alpha;
  // the centre table serves X3 faces wherever the metric does not depend on x3
  if (DIR == 3 && MF != FORM_NULLV && (MF != FORM_FULL || !G.face[2])) {
    const uint32_t t = (uint32_t)cen_index(G, k, j, i);
    auto comp = [&](int n) { return ldc32(G.cen, (int64_t)n * (uint32_t)G.ncen, t); };
    load_metric<MF, CG_GCON, CG_ALPHA>(comp, g, gc0, alpha);
    if (MF != FORM_FLAT) {
      gdd = comp(CG_GCON + 15);
      sg = comp(CG_SG);
    }
  } else {
    const int d = DIR - 1;
    const uint32_t t = (uint32_t)(((G.has3d ? k : 0) * G.fj[d] + j) * G.fi[d] + i);
    auto comp = [&](int n) { return ldc32(G.face[d], (int64_t)n * (uint32_t)G.nface[d], t); };
    load_metric<MF, FG_GCON0, FG_ALPHA>(comp, g, gc0, alpha);
    if (MF != FORM_FLAT) {
      gdd = comp(FG_GCONDD);
      sg = comp(FG_SG);
    }
  }
  double *const al = alfven[b * 3 + (DIR - 1)];
  const uint32_t id32 = (uint32_t)id;
  // a singular face metric (polar axis; its table entry holds alpha = 0)
  // has zero flux and wave speed
  if (MF != FORM_FLAT && alpha == 0.0) {
    st32(al, id32, 0.0);
#pragma unroll
    for (int q = 0; q < NC; ++q) st32(F.flux[DIR - 1][b * NC + q], id32, 0.0);
    return;
  }
  const double gam = C.ph.gamma;
  St sl, sr;
  calc_state<MF, HB>(pl, g, gc0, alpha, sl);
  calc_state<MF, HB>(pr, g, gc0, alpha, sr);
  double vmaxL, vminL, vmaxR, vminR;
  fast_ms<DIR, MF, HB>(gam, pl, sl, gc0[0], gc0[DIR], gdd, vmaxL, vminL);
  fast_ms<DIR, MF, HB>(gam, pr, sr, gc0[0], gc0[DIR], gdd, vmaxR, vminR);
  const double cmax = fabs(kmax(kmax(0., vmaxL), vmaxR));
  const double cmin = fabs(kmax(kmax(0., -vminL), -vminR));
  const double cc = kmax(cmax, cmin);
  st32(al, id32, cc);
  double UL[NPRIM], UR[NPRIM], FL[NPRIM], FR[NPRIM];
  contravariant_flux<0, HB>(gam, pl, sl, sg, UL);
  contravariant_flux<0, HB>(gam, pr, sr, sg, UR);
  contravariant_flux<DIR, HB>(gam, pl, sl, sg, FL);
  contravariant_flux<DIR, HB>(gam, pr, sr, sg, FR);
  // The fluxes go past L2: the update reads them after the last sweep, and
  // until then the stencils' P has a better use for the lines (3-D torus
  // 256x128x128: 3.94 -> 3.83 ms per cycle; with the update's U stored the same
  // way 3.81 ms; loads of U_init or stores of P that way gain nothing).
  const double den = cmax + cmin + 1e-20, rden = quot(1.0, den);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int s = slot_of<HB, HK>(q);
    double f;
    if (RS == PANGU_RIEMANN_LAXF)
      f = 0.5 * (FL[s] + FR[s] - cc * (UR[s] - UL[s]));
    else
      f = div_by(cmax * FL[s] + cmin * FR[s] - cmax * cmin * (UR[s] - UL[s]), den, rden);
    stnt32(F.flux[DIR - 1][b * NC + q], id32, f);
  }
}

// Face (k, j, i) of the sweep along DIR.
template <int DIR, int LIM, int RS, bool HB, bool HK, int MF>
__device__ __forceinline__ void sweep_face(const KCtx &C, const KFields &F, double *const *alfven, int b,
                                           int k, int j, int i) {
  const DevBlock &B = C.blk[b];
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t st = (DIR == 1) ? 1 : (DIR == 2 ? sj : sk);
  const int64_t id = k * sk + j * sj + i;
  constexpr int NC = ncomp<HB, HK>();
  double pl[NPRIM], pr[NPRIM];
#pragma unroll
  for (int s = 0; s < NPRIM; ++s) {
    pl[s] = 0.0;
    pr[s] = 0.0;
  }
  // Every stencil value of every variable is loaded before the first
  // reconstruction, so a wavefront waits for memory once rather than once
  // per variable (the compiler keeps the loads of an unrolled per-variable
  // loop behind each variable's arithmetic).  The peak register use stays in
  // the face physics.
  constexpr int NS = (LIM == PANGU_LIMITER_PPM4) ? 6 : 4;  // offsets -NS/2 .. NS/2 - 1
  double v[NC][NS];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const double *a = F.prim[b * NC + q];
#pragma unroll
    for (int n = 0; n < NS; ++n)
      // x1 neighbours fold into the load's immediate offset; x2/x3 offsets
      // (a row, a plane) into the scalar base
      v[q][n] = DIR == 1 ? glb(a)[id + (n - NS / 2)] : ld32(a, (n - NS / 2) * st, (uint32_t)id);
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int s = slot_of<HB, HK>(q);
    double t0, t1;
    if (LIM == PANGU_LIMITER_PPM4) {
      recon_ppm4(v[q][0], v[q][1], v[q][2], v[q][3], v[q][4], pl[s], t0);
      recon_ppm4(v[q][1], v[q][2], v[q][3], v[q][4], v[q][5], t1, pr[s]);
    } else {
      recon_mc(v[q][0], v[q][1], v[q][2], pl[s], t0);
      recon_mc(v[q][1], v[q][2], v[q][3], t1, pr[s]);
    }
  }
  face_flux<DIR, RS, HB, HK, MF>(C, F, alfven, b, k, j, i, pl, pr);
}

}  // namespace pangu
