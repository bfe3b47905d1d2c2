// Every flux sweep of a stage in one launch, with the stage's ghost exchange
// as a passenger.
#include <hip/hip_runtime.h>

#include "common.h"
#include "flux_dev.h"
#include "halo_dev.h"
#include "kernels.h"
#include "launch_host.h"
#include "tiles_dev.h"

namespace pangu {

// What a launch holds: the face ranges of the nd active directions, and the
// ghost exchange of another container (ghosts.ntiles = 0: none).
struct SweepSet {
  Range3 R[3];
  int n8[4];   // tiles per XCD of each direction, then of the exchange
  int nd;
  int run;     // consecutive tiles of one direction on an XCD
  int sweeps;  // workgroups per XCD that hold sweep tiles; the exchange's follow
  Items ghosts;
  KFields X;
  double *const *flag;
  const int *nbr;
};

// The sweeps read the same P and write different arrays, so nothing orders
// them, and one launch fills the chip where a direction alone leaves CUs
// empty (a 256^2 block has 264 workgroups per direction) and starts once.
// Workgroup L goes to XCD L mod 8, which owns an eighth of each direction's
// tiles.  On an XCD the directions take turns in runs of kRun tiles: X2 and X3
// then find the P that X1 read still cached (256 tiles of ten components are
// 5 MB, 42 MB over the XCDs, against 256 MB of last-level cache), while most
// of the XCD's CUs run one direction's code at a time.  The exchange comes
// last and fills the sweeps' tail.  Sweeps one by one, in one launch in turn,
// in runs of 1, 64, 256 and 512 tiles: 4.14, 4.11, 4.04, 4.03, 4.00 and 4.02 ms
// per cycle on the 3-D torus 256x128x128.  Exchange tiles taken in turn with
// the sweeps': 4.75 ms (a light kernel's workgroups at the sweeps' register
// count, three wavefronts per SIMD).  Small meshes gain most: sweeps one by one ->
// merged -> with the exchange, Orszag-Tang 256^2 97 -> 86 -> 80 us, eight
// 32x16x16 torus blocks 169 -> 141 -> 132 us, ensemble of 20 meshes 458 -> 424 ->
// 412 us, 2-D torus 512x256 196 -> 181 -> 174 us.
constexpr int kRun = 256;

template <int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256) void k_sweeps(KCtx C, KFields F, double *const *alfven, SweepSet S) {
  const int L = (int)blockIdx.x, m = L >> 3;
  int kind = 3, r = m - S.sweeps;
  if (r < 0) {
    const int turn = m / (S.nd * S.run), in = m - turn * S.nd * S.run;
    kind = in / S.run;
    r = turn * S.run + in - kind * S.run;
  }
  if (r >= S.n8[kind]) return;
  const int T = (L & 7) * S.n8[kind] + r;
  int b, k, j, i;
  if (kind == 3) {
    if (T >= S.ghosts.ntiles) return;
    decode_item_at(S.ghosts, T, b, k);
    exchange_cell<ncomp<HB, HK>()>(C, S.X, S.flag, S.nbr, b, k);
    return;
  }
  if (T >= S.R[kind].ntiles || !decode_tile_at(C, S.R[kind], T, b, k, j, i)) return;
  if (kind == 0)
    sweep_face<1, LIM, RS, HB, HK, MF>(C, F, alfven, b, k, j, i);
  else if (kind == 1)
    sweep_face<2, LIM, RS, HB, HK, MF>(C, F, alfven, b, k, j, i);
  else
    sweep_face<3, LIM, RS, HB, HK, MF>(C, F, alfven, b, k, j, i);
}

// ===================================================================== host
bool sweeps_merge(const LaunchCtx &L) {
  const int *t = &L.tile[PANGU_KF_FLUX_X1];
  return !L.clock && !L.share_x1 && !L.pair_flux && !L.march_depth[0] && !L.march_depth[1] && t[0] == t[1] &&
         t[1] == t[2] && L.face[0].ntiles > 0 && (L.k.ndim < 2 || L.face[1].ntiles > 0);
}

template <int LIM, int RS, bool HB, bool HK>
static void launch_form(const LaunchCtx &L, const KFields &F, double *const *alfven, const SweepSet &S, dim3 g,
                        dim3 wg, hipStream_t s) {
  const int mf = metric_form(L.metric);
  if (mf == FORM_POLOIDAL)
    hipLaunchKernelGGL((k_sweeps<LIM, RS, HB, HK, FORM_POLOIDAL>), g, wg, 0, s, L.k, F, alfven, S);
  else if (mf == FORM_FLAT)
    hipLaunchKernelGGL((k_sweeps<LIM, RS, HB, HK, FORM_FLAT>), g, wg, 0, s, L.k, F, alfven, S);
  else
    hipLaunchKernelGGL((k_sweeps<LIM, RS, HB, HK, FORM_NULLV>), g, wg, 0, s, L.k, F, alfven, S);
}
template <int LIM, int RS>
static void launch_fields(const LaunchCtx &L, const KFields &F, double *const *alfven, const SweepSet &S,
                          dim3 g, dim3 wg, hipStream_t s) {
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  if (hb && hk)
    launch_form<LIM, RS, true, true>(L, F, alfven, S, g, wg, s);
  else if (hb)
    launch_form<LIM, RS, true, false>(L, F, alfven, S, g, wg, s);
  else if (hk)
    launch_form<LIM, RS, false, true>(L, F, alfven, S, g, wg, s);
  else
    launch_form<LIM, RS, false, false>(L, F, alfven, S, g, wg, s);
}

int launch_sweeps(const LaunchCtx &L, const KFields &F, double *const *alfven, const ExchangeArgs *ex,
                  hipStream_t s) {
  SweepSet S;
  S.nd = 0;
  int most = 0;
  for (int d = 0; d < 3; ++d) {
    S.R[d] = family_range(L, 2 + d, L.face[d], PANGU_KF_FLUX_X1 + d);
    S.n8[d] = (S.R[d].ntiles + 7) / 8;
    if (S.R[d].ntiles > 0) S.nd = d + 1;
    most = S.n8[d] > most ? S.n8[d] : most;
  }
  S.ghosts = Items{nullptr, nullptr, 0};
  S.X = F;
  S.flag = nullptr;
  S.nbr = nullptr;
  if (ex) {
    S.ghosts = L.ghosts;
    S.X = ex->F;
    S.flag = ex->flag;
    S.nbr = ex->nbr;
  }
  S.n8[3] = (S.ghosts.ntiles + 7) / 8;
  S.run = most < kRun ? most : kRun;
  S.sweeps = S.nd * S.run * ((most + S.run - 1) / S.run);
  const dim3 g((unsigned)(8 * (S.sweeps + S.n8[3]))), wg(S.R[0].tile);
  if (L.limiter == PANGU_LIMITER_PPM4) {
    if (L.riemann == PANGU_RIEMANN_HLL)
      launch_fields<PANGU_LIMITER_PPM4, PANGU_RIEMANN_HLL>(L, F, alfven, S, g, wg, s);
    else
      launch_fields<PANGU_LIMITER_PPM4, PANGU_RIEMANN_LAXF>(L, F, alfven, S, g, wg, s);
  } else {
    if (L.riemann == PANGU_RIEMANN_HLL)
      launch_fields<PANGU_LIMITER_MC, PANGU_RIEMANN_HLL>(L, F, alfven, S, g, wg, s);
    else
      launch_fields<PANGU_LIMITER_MC, PANGU_RIEMANN_LAXF>(L, F, alfven, S, g, wg, s);
  }
  return PG_CHECK_LAUNCH();
}

}  // namespace pangu
