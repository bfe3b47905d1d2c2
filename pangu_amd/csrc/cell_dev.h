// What the cell kernels of kernels.hip and flux.hip share: the packed field
// order and the loads of the geometry tables.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "physics_dev.h"

namespace pangu {

// Packed component q -> slot, for the enabled field set
// (package_registration.cc:84-96).
template <bool HB, bool HK>
__device__ __forceinline__ constexpr int slot_of(int q) {
  return q < 5 ? q : (HB ? (q < 8 ? q : (q == 8 ? ENT : KEL)) : (q == 5 ? ENT : KEL));
}
template <bool HB, bool HK>
__device__ __forceinline__ constexpr int ncomp() {
  return 6 + (HB ? 3 : 0) + (HK ? 1 : 0);
}
template <bool HB>
__device__ __forceinline__ constexpr int ient() {
  return HB ? 8 : 5;
}
template <bool HB>
__device__ __forceinline__ constexpr int ikel() {
  return HB ? 9 : 6;
}

__device__ __forceinline__ int64_t cen_index(const DevGeo &G, int k, int j, int i) {
  return ((int64_t)(G.has3d ? k : 0) * G.nj + j) * G.ni + i;
}

static_assert(CG_GCOV == 0 && FG_GCOV == 0 && (int)CG_NUL == (int)FG_NUL, "both tables keep gcov alike");

// gcov = eta + (xi l_r) l_c as the host forms it; comp(n) loads component n.
template <class LD>
__device__ __forceinline__ void gcov_from_null(LD comp, double g[16]) {
  const double xi = comp(CG_NUL), l[4] = {1.0, comp(CG_NUL + 1), comp(CG_NUL + 2), comp(CG_NUL + 3)};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double t = r ? xi * l[r] : xi;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double u = c ? t * l[c] : t;
      g[4 * r + c] = r != c ? u : (r ? 1.0 : -1.0) + u;
    }
  }
}

// gcov of a table entry of any metric (nullv: DevGeo's), for readers that are
// not compiled per form.
template <class LD>
__device__ __forceinline__ void load_gcov(LD comp, int nullv, double g[16]) {
  if (nullv) {
    gcov_from_null(comp, g);
  } else {
#pragma unroll
    for (int n = 0; n < 16; ++n) g[n] = comp(n);
  }
}

// gcov, g^{0m} and the lapse of a table entry, as far as form MF leaves them
// open; the symmetric partner of a loaded entry shares its register.
// comp(n) loads component n; GCON0 and ALPHA are the table's component
// numbers of g^{00} and of 1/sqrt(-g^{00}).
template <int MF, int GCON0, int ALPHA, class LD>
__device__ __forceinline__ void load_metric(LD comp, double g[16], double gc0[4], double &alpha) {
  if (MF == FORM_FLAT) {
#pragma unroll
    for (int n = 0; n < 16; ++n) g[n] = (n % 5) ? 0.0 : (n ? 1.0 : -1.0);
#pragma unroll
    for (int n = 0; n < 4; ++n) gc0[n] = n ? 0.0 : -1.0;
    alpha = 1.0;
    return;
  }
  if (MF == FORM_NULLV) {
    gcov_from_null(comp, g);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int slot = g_slot<MF>(r, c);
        g[4 * r + c] = !g_open<MF>(r, c) ? 0.0 : (slot < 4 * r + c ? g[slot] : comp(slot));
      }
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) gc0[n] = g0_open<MF>(n) ? comp(GCON0 + n) : 0.0;
  alpha = comp(ALPHA);
}

// Loads of the centre table.
struct CenLoad {
  double g[16], gc0[4], alpha, sg;
};
template <int MF = FORM_FULL>
__device__ __forceinline__ void load_cen_state(const DevGeo &G, int64_t t, CenLoad &m) {
  const double *c = G.cen;
  const int64_t s = G.ncen;
  const uint32_t t32 = (uint32_t)t;
  auto comp = [&](int n) { return ldc32(c, n * s, t32); };
  load_metric<MF, CG_GCON, CG_ALPHA>(comp, m.g, m.gc0, m.alpha);
  m.sg = MF == FORM_FLAT ? 1.0 : comp(CG_SG);
}

}  // namespace pangu
