// Host side of the tile launches: grids, per-family ranges, the launch check
// and the per-launch clock mark.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "tiles_dev.h"

namespace pangu {

// Grid of a tile launch, padded to a multiple of the 8 XCDs.
inline dim3 tile_grid(const Range3 &R) { return dim3((unsigned)(((R.ntiles + 7) / 8) * 8)); }
static const dim3 kTile(TILE, 1, 1);

// Range of a launch of kernel family fam over base range id (0 interior,
// 1 entire, 2..4 the faces, 5 CT) in that family's tile size and order.
inline Range3 family_range(const LaunchCtx &L, int id, const Range3 &base, int fam) {
  const int t = L.tile[fam];
  Range3 R = (t == 128) ? L.small[id][0] : (t == 64) ? L.small[id][1] : base;
  R.order = L.order[fam];
  return R;
}

// Recovery with the learned start of W or, without a model, as a persistent
// work queue (recovery_options.hip); heat only where there is K_e.
void launch_recover_option(const LaunchCtx &L, const KFields &F, const SharedTabs &S, int rec, bool heat,
                           const MlpFrag *W, const Range3 &R, hipStream_t s, const UpdArgs *upd);
// The sweep along dir in one of its other forms (flux_options.hip).  0: the
// plain form is asked for; 1: launched; -1: nothing to launch.
int launch_sweep_option(const LaunchCtx &L, int dir, const KFields &F, double *const *alfven, hipStream_t s);

#define PG_CHECK_LAUNCH() (hipGetLastError() == hipSuccess ? 0 : -2)
#define TICK(name) \
  if (L.clock) (void)L.clock->mark(name, s)

}  // namespace pangu
