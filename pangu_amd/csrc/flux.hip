// gfx950 kernels of FixPrimitive, the conserved state and the flux sweeps
// (FP64 vector ALU).  Thread mapping: see kernels.hip.
#include <hip/hip_runtime.h>

#include "cell_dev.h"
#include "common.h"
#include "fix_dev.h"
#include "flux_dev.h"
#include "kernels.h"
#include "launch_host.h"
#include "physics_dev.h"
#include "tiles_dev.h"

namespace pangu {

template <int MF, bool FIX, bool CONS, bool HB, bool HK>
__global__ __launch_bounds__(256) void k_fix_cons(KCtx C, KFields F, uint8_t *const *mask, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  fix_cons_cell<MF, FIX, CONS, HB, HK>(C, F, mask, b, k, j, i, true, nullptr);
}

// ------------------------------------------------------------- flux sweep
template <int DIR, int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256) void k_flux(KCtx C, KFields F, double *const *alfven, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  sweep_face<DIR, LIM, RS, HB, HK, MF>(C, F, alfven, b, k, j, i);
}

// ===================================================================== host
int launch_fix_cons(const LaunchCtx &L, const KFields &F, uint8_t *const *mask, bool fix, bool cons,
                    hipStream_t s) {
  const Range3 R = fix ? family_range(L, 1, L.entire, PANGU_KF_FIX_CONS)
                       : family_range(L, 0, L.interior, PANGU_KF_FIX_CONS);
  if (R.ntiles == 0) return 0;
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  const int mf = metric_form(L.metric);
#define FC(FX, CS, HB_, HK_)                                                                          \
  if (mf == FORM_POLOIDAL)                                                                            \
    hipLaunchKernelGGL((k_fix_cons<FORM_POLOIDAL, FX, CS, HB_, HK_>), g, wg, 0, s, L.k, F, mask, R);  \
  else if (mf == FORM_FLAT)                                                                           \
    hipLaunchKernelGGL((k_fix_cons<FORM_FLAT, FX, CS, HB_, HK_>), g, wg, 0, s, L.k, F, mask, R);      \
  else                                                                                                \
    hipLaunchKernelGGL((k_fix_cons<FORM_NULLV, FX, CS, HB_, HK_>), g, wg, 0, s, L.k, F, mask, R)
#define FC2(FX, CS)                                \
  if (hb && hk) { FC(FX, CS, true, true); }        \
  else if (hb) { FC(FX, CS, true, false); }        \
  else if (hk) { FC(FX, CS, false, true); }        \
  else { FC(FX, CS, false, false); }
  if (fix && cons) {
    FC2(true, true)
  } else if (fix) {
    FC2(true, false)
  } else {
    FC2(false, true)
  }
#undef FC2
#undef FC
  TICK(fix && cons ? "fix_cons" : fix ? "fix_primitive" : "conservative");
  return PG_CHECK_LAUNCH();
}

template <int DIR>
static void flux_dir(const LaunchCtx &L, const KFields &F, double *const *alfven, hipStream_t s) {
  const int option = launch_sweep_option(L, DIR, F, alfven, s);
  const Range3 R = family_range(L, 1 + DIR, L.face[DIR - 1], PANGU_KF_FLUX_X1 + DIR - 1);
  if (option < 0 || (option == 0 && R.ntiles == 0)) return;
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  const int lim = L.limiter, rs = L.riemann, mf = metric_form(L.metric);
#define FL(LIM, RS, HB_, HK_)                                                                      \
  if (mf == FORM_POLOIDAL)                                                                        \
    hipLaunchKernelGGL((k_flux<DIR, LIM, RS, HB_, HK_, FORM_POLOIDAL>), g, wg, 0, s, L.k, F, alfven, R); \
  else if (mf == FORM_FLAT)                                                                       \
    hipLaunchKernelGGL((k_flux<DIR, LIM, RS, HB_, HK_, FORM_FLAT>), g, wg, 0, s, L.k, F, alfven, R); \
  else                                                                                            \
    hipLaunchKernelGGL((k_flux<DIR, LIM, RS, HB_, HK_, FORM_NULLV>), g, wg, 0, s, L.k, F, alfven, R)
#define FL2(LIM, RS)                         \
  if (hb && hk) { FL(LIM, RS, true, true); } \
  else if (hb) { FL(LIM, RS, true, false); } \
  else if (hk) { FL(LIM, RS, false, true); } \
  else { FL(LIM, RS, false, false); }
  if (option != 0) {
    // launched there
  } else if (lim == PANGU_LIMITER_PPM4 && rs == PANGU_RIEMANN_LAXF) {
    FL2(PANGU_LIMITER_PPM4, PANGU_RIEMANN_LAXF)
  } else if (lim == PANGU_LIMITER_PPM4) {
    FL2(PANGU_LIMITER_PPM4, PANGU_RIEMANN_HLL)
  } else if (rs == PANGU_RIEMANN_LAXF) {
    FL2(PANGU_LIMITER_MC, PANGU_RIEMANN_LAXF)
  } else {
    FL2(PANGU_LIMITER_MC, PANGU_RIEMANN_HLL)
  }
#undef FL2
#undef FL
  TICK(DIR == 1 ? "flux_x1" : DIR == 2 ? "flux_x2" : "flux_x3");
}

int launch_fluxes_23(const LaunchCtx &L, const KFields &F, double *const *alfven, hipStream_t s) {
  flux_dir<2>(L, F, alfven, s);
  flux_dir<3>(L, F, alfven, s);
  return PG_CHECK_LAUNCH();
}

int launch_fluxes(const LaunchCtx &L, const KFields &F, double *const *alfven, hipStream_t s) {
  if (sweeps_merge(L)) return launch_sweeps(L, F, alfven, nullptr, s);
  flux_dir<1>(L, F, alfven, s);
  flux_dir<2>(L, F, alfven, s);
  flux_dir<3>(L, F, alfven, s);
  return PG_CHECK_LAUNCH();
}

}  // namespace pangu
