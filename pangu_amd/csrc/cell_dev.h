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

// Loads of the centre table.
struct CenLoad {
  double g[16], gc0[4], alpha, sg;
};
__device__ __forceinline__ void load_cen_state(const DevGeo &G, int64_t t, CenLoad &m) {
  const double *c = G.cen;
  const int64_t s = G.ncen;
  const uint32_t t32 = (uint32_t)t;
#pragma unroll
  for (int n = 0; n < 16; ++n) m.g[n] = ldc32(c, (CG_GCOV + n) * s, t32);
#pragma unroll
  for (int n = 0; n < 4; ++n) m.gc0[n] = ldc32(c, (CG_GCON + n) * s, t32);
  m.alpha = ldc32(c, CG_ALPHA * s, t32);
  m.sg = ldc32(c, CG_SG * s, t32);
}

}  // namespace pangu
