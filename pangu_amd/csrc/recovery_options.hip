// Recovery kernels that a run asks for: the persistent work queue and the
// learned start.  (A file of their own: a program that never asks does not
// load them.)
#include <hip/hip_runtime.h>
#include <float.h>

#include "cell_dev.h"
#include "common.h"
#include "kernels.h"
#include "launch_host.h"
#include "mlp_dev.h"
#include "physics_dev.h"
#include "recovery_dev.h"
#include "tiles_dev.h"
#include "update_dev.h"

namespace pangu {

// Persistent form of k_recover: a grid no larger than what the GPU holds
// at once pulls tiles from a queue (queue[0]: next tile, queue[1]:
// workgroups done) until every tile is taken; the last workgroup out resets
// the queue for the next launch on the stream, so a captured graph replays
// it without a memset.  Tiles carry no dependencies, so no workgroup ever
// waits for another.  Same cells, same arithmetic: identical results.
template <int MF, int REC, bool HB, bool HK, bool HEAT>
__global__ __launch_bounds__(256) void k_recover_queue(KCtx C, KFields F, SharedTabs S, Range3 R,
                                                       unsigned *queue) {
  __shared__ int tile_sh;
  for (;;) {
    if (threadIdx.x == 0) tile_sh = (int)atomicAdd(&queue[0], 1u);
    __syncthreads();
    const int T = tile_sh;
    __syncthreads();  // every thread has read the tile before the next pull
    if (T >= R.ntiles) break;
    int b, k, j, i;
    if (decode_tile_at(C, R, T, b, k, j, i)) recover_cell<MF, REC, HB, HK, HEAT>(C, F, S, b, k, j, i);
  }
  if (threadIdx.x == 0 && atomicAdd(&queue[1], 1u) == gridDim.x - 1) {
    atomicExch(&queue[0], 0u);
    atomicExch(&queue[1], 0u);
  }
}

// Kastaun recovery with the learned starting bracket (and, when HEAT, the
// electron heating): k_recover<1, ...> whose wavefronts that hold a cell
// passing the gate (its previous recovery took at least S.gate
// false-position steps) run the network on the matrix cores inside the
// wavefront (wave_mlp); every cell of such a wavefront then starts the
// search from the prediction (kastaun_guess_k), the others search [0, 1]
// as k_recover does.  Status, iteration and field outputs are those of
// k_recover; the recovered state agrees with it to the solver tolerance
// (another false-position path to a root of the same function), not bit for
// bit.
template <int MF, bool HB, bool HK>
__device__ __forceinline__ int learned_setup(const KCtx &C, const KFields &F, const DevGeo &G, int64_t t,
                                             int b, int64_t id, KastaunIn &kin) {
  constexpr int NC = ncomp<HB, HK>();
  const int64_t ns = G.ncen;
  CenMetric m;
  auto comp = [&](int n) { return ldc32(G.cen, (int64_t)n * ns, (uint32_t)t); };
  if (MF == FORM_NULLV)
    gcov_from_null(comp, m.gcov);
  else
    load_gcov(comp, 0, m.gcov);
#pragma unroll
  for (int n = 0; n < 16; ++n) m.gcon[n] = comp(CG_GCON + n);
  m.lapse = ldc32(G.cen, (int64_t)CG_LAPSE * ns, (uint32_t)t);
  const double aos = ldc32(G.cen, (int64_t)CG_ALPHA * ns, (uint32_t)t) * (1.0 / ldc32(G.cen, (int64_t)CG_SG * ns, (uint32_t)t));
  const double *const *cons = F.cons + (int64_t)b * NC;
  const double c_rho = glb(cons[0])[id], c_eny = glb(cons[1])[id];
  double U[9];
  U[RHO] = aos * c_rho;
  U[ENY] = aos * (c_eny - c_rho);
  U[UX1] = aos * glb(cons[2])[id];
  U[UX2] = aos * glb(cons[3])[id];
  U[UX3] = aos * glb(cons[4])[id];
#pragma unroll
  for (int a = 0; a < 3; ++a) U[BX1 + a] = HB ? aos * glb(cons[5 + a])[id] : 0.0;
  U[ENT] = aos * glb(cons[ient<HB>()])[id];
  return kastaun_setup(U, m, kin);
}

// UPD 1 or 2: the cell's update (k_div_update mode 4; 2 with the source)
// runs first, as in k_update_recover; the recovery then reads the U this
// thread has just stored.
template <int MF, bool HB, bool HK, bool HEAT, int UPD>
__global__ __launch_bounds__(256) void k_recover_learned(KCtx C, KFields F, SharedTabs S, MlpFrag W,
                                                         Range3 R, UpdArgs A) {
  int b = 0, k = 0, j = 0, i = 0;
  const bool cell = decode_tile(C, R, b, k, j, i);  // false on the whole workgroup past the range
  if (UPD && cell)
    div_update_cell<4, UPD == 2 ? MF : FORM_FLAT, HB, HK, HB>(C, A.F0, A.Finit, F, nullptr, A.dt_dev, A.beta, A.bdt_host, b,
                                             k, j, i, nullptr);
  const int lane = threadIdx.x & 63;
  constexpr int NC = ncomp<HB, HK>();
  const Phys &P = C.ph;
  const DevBlock &B = C.blk[cell ? b : 0];
  const DevGeo &G = C.geo[B.geo];
  const int64_t id = cell ? ((int64_t)k * B.n[1] + j) * B.n[0] + i : 0;
  const int64_t t = cell ? cen_index(G, k, j, i) : 0;
  const bool active =
      cell && !(P.metric == PANGU_METRIC_CKS && ldc32(G.cen, (int64_t)CG_RAD * G.ncen, (uint32_t)t) < P.r_excise);
  // The workgroup votes on the previous iteration counts alone, before any
  // other load: a workgroup with no cell passing the gate then runs as
  // k_recover<1> does, with no further barrier.  The network's cost is per
  // wavefront, so a wavefront that runs it for a gated cell serves every
  // cell of it with a valid setup.
  int prev = 0;
  if (active && S.iters) prev = glb(S.iters[b])[id];
  const bool gated = active && S.iters && prev >= S.gate;
  KastaunIn kin;
  int setup = -1;
  double guess = -1.0;
  __shared__ MlpLds lds;
  // every thread of the workgroup reaches the vote (no early return above)
  if (__syncthreads_or(gated)) {
    mlp_stage(W, lds, threadIdx.x, blockDim.x);
    if (active) setup = learned_setup<MF, HB, HK>(C, F, G, t, b, id, kin);
    __syncthreads();
    const bool want = setup == 0;
    if (__ballot(gated && want)) {  // uniform over the wavefront: all 64 lanes run the network
      float x[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      if (want) {
        float f[5];
        c2p_features(kin, f);
#pragma unroll
        for (int q = 0; q < 5; ++q) x[q] = bf2f(f2bf((f[q] - W.mean[q]) / W.dev[q]));
      }
      const float z = wave_mlp(lds, W.b4[0], x, lane);
      if (want) guess = (double)(1.0f / (1.0f + expf(-z)));
      // the setup is recomputed from memory (same inputs, same bits)
      // instead of being held in registers across the network
      __asm__ volatile("" ::: "memory");
      if (active) setup = learned_setup<MF, HB, HK>(C, F, G, t, b, id, kin);
    }
  } else if (active) {
    setup = learned_setup<MF, HB, HK>(C, F, G, t, b, id, kin);
  }
  if (!cell) return;
  Arr32<double> pp[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) pp[q] = Arr32<double>{F.prim[b * NC + q]};
  if (!active) {
    if (S.status) glb(S.status[b])[id] = -1;
    if (S.iters) glb(S.iters[b])[id] = 0;
  } else {
    double bnew[3] = {0.0, 0.0, 0.0};
    if (HB) {
      const double isg = 1.0 / ldc32(G.cen, (int64_t)CG_SG * G.ncen, (uint32_t)t);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        bnew[a] = glb(F.cons[b * NC + 5 + a])[id] * isg;
        pp[5 + a][id] = bnew[a];
      }
    }
    double Ph[9];
    double mu = 0.0;
    int st, it = 0;
    if (setup != 0) {
      st = setup;
    } else {
      // one code path: without a guess (-1) kastaun_guess_k searches [0, 1]
      // exactly as kastaun_plain_k does
      int ev = 0;
      st = kastaun_guess_k(kin, P.gamma, Ph, guess, S.delta, it, ev, &mu);
    }
    if (S.root) glb(S.root[b])[id] = (st == 0) ? mu : __builtin_nan("");
    if (S.status) glb(S.status[b])[id] = st;
    if (S.iters) glb(S.iters[b])[id] = it;
    if (st == 0) {
      pp[0][id] = Ph[RHO];
      pp[1][id] = Ph[ENY];
      pp[2][id] = Ph[UX1];
      pp[3][id] = Ph[UX2];
      pp[4][id] = Ph[UX3];
    }
    if (HEAT && HK) {
      // as recover_cell: the heating takes the primitives just written from
      // registers (a failed cell keeps its previous ones, from memory)
      double hp[NPRIM];
#pragma unroll
      for (int q = 0; q < NPRIM; ++q) hp[q] = 0.0;
      if (st == 0) {
        hp[RHO] = Ph[RHO];
        hp[ENY] = Ph[ENY];
        hp[UX1] = Ph[UX1];
        hp[UX2] = Ph[UX2];
        hp[UX3] = Ph[UX3];
      } else {
        hp[RHO] = pp[0][id];
        hp[ENY] = pp[1][id];
        hp[UX1] = pp[2][id];
        hp[UX2] = pp[3][id];
        hp[UX3] = pp[4][id];
      }
      if (HB) {
#pragma unroll
        for (int a = 0; a < 3; ++a) hp[BX1 + a] = bnew[a];
      }
      hp[ENT] = pp[ient<HB>()][id];
      heat_vals<MF, HB, HK>(C, F, G, t, b, id, pp, hp);
      return;
    }
  }
  if (HEAT && HK) heat_cell<MF, HB, HK>(C, F, G, t, b, id, pp);
}

// The 1Dvsq recovery with the learned start (and, when HEAT, the heating):
// the vote, the staging and the in-wave network of k_recover_learned, on
// the same features (the Kastaun invariants of the cell's U and metric),
// predicting z = log u^2; every cell of a wavefront that ran the network
// then starts its Newton iteration from v^2 = u^2 / (1 + u^2) =
// logistic(z) instead of the previous primitives' v^2.  Everything else is
// recover_cell<2>: the result agrees with k_recover<2> to the Newton
// tolerance, not bit for bit.
template <int MF, bool HB, bool HK, bool HEAT, int UPD>
__global__ __launch_bounds__(256) void k_recover_learned_vsq(KCtx C, KFields F, SharedTabs S, MlpFrag W,
                                                             Range3 R, UpdArgs A) {
  int b = 0, k = 0, j = 0, i = 0;
  const bool cell = decode_tile(C, R, b, k, j, i);  // false on the whole workgroup past the range
  if (UPD && cell)
    div_update_cell<4, UPD == 2 ? MF : FORM_FLAT, HB, HK, HB>(C, A.F0, A.Finit, F, nullptr, A.dt_dev, A.beta, A.bdt_host, b,
                                             k, j, i, nullptr);
  const int lane = threadIdx.x & 63;
  const Phys &P = C.ph;
  const DevBlock &B = C.blk[cell ? b : 0];
  const DevGeo &G = C.geo[B.geo];
  const int64_t id = cell ? ((int64_t)k * B.n[1] + j) * B.n[0] + i : 0;
  const int64_t t = cell ? cen_index(G, k, j, i) : 0;
  const bool active =
      cell && !(P.metric == PANGU_METRIC_CKS && ldc32(G.cen, (int64_t)CG_RAD * G.ncen, (uint32_t)t) < P.r_excise);
  int prev = 0;
  if (active && S.iters) prev = glb(S.iters[b])[id];
  const bool gated = active && S.iters && prev >= S.gate;
  double x0 = -1.0;
  __shared__ MlpLds lds;
  // every thread of the workgroup reaches the vote (no early return above)
  if (__syncthreads_or(gated)) {
    mlp_stage(W, lds, threadIdx.x, blockDim.x);
    KastaunIn kin;
    const int setup = active ? learned_setup<MF, HB, HK>(C, F, G, t, b, id, kin) : -1;
    __syncthreads();
    const bool want = setup == 0;
    if (__ballot(gated && want)) {  // uniform over the wavefront: all 64 lanes run the network
      float x[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      if (want) {
        float f[5];
        c2p_features(kin, f);
#pragma unroll
        for (int q = 0; q < 5; ++q) x[q] = bf2f(f2bf((f[q] - W.mean[q]) / W.dev[q]));
      }
      const float z = wave_mlp(lds, W.b4[0], x, lane);
      if (want) x0 = (double)(1.0f / (1.0f + expf(-z)));
    }
  }
  if (!cell) return;
  recover_cell<MF, 2, HB, HK, HEAT>(C, F, S, b, k, j, i, x0);
}

// ===================================================================== host
// Grid of a persistent kernel: the workgroups the GPU holds at once (at
// most ntiles), so every workgroup runs from the start.
template <typename K>
static int resident_groups(K kernel, int threads, int ntiles) {
  int dev = 0, per_cu = 0, ncu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 1;
  const int64_t n = (int64_t)(per_cu > 0 ? per_cu : 1) * (ncu > 0 ? ncu : 1);
  return (int)(n < ntiles ? n : ntiles);
}

template <int MF, bool HB, bool HK, bool HEAT>
static void launch_learned(const LaunchCtx &L, const KFields &F, const SharedTabs &S, const MlpFrag &W,
                           const Range3 &R, dim3 g, dim3 wg, hipStream_t s, const UpdArgs *upd) {
  const UpdArgs A = upd ? *upd : UpdArgs{};
  const int u = !upd ? 0 : (L.metric != PANGU_METRIC_MINKOWSKI ? 2 : 1);
  if (W.kind == 0) {
    if (u == 2)
      hipLaunchKernelGGL((k_recover_learned<MF, HB, HK, HEAT, 2>), g, wg, 0, s, L.k, F, S, W, R, A);
    else if (u == 1)
      hipLaunchKernelGGL((k_recover_learned<MF, HB, HK, HEAT, 1>), g, wg, 0, s, L.k, F, S, W, R, A);
    else
      hipLaunchKernelGGL((k_recover_learned<MF, HB, HK, HEAT, 0>), g, wg, 0, s, L.k, F, S, W, R, A);
  } else {
    if (u == 2)
      hipLaunchKernelGGL((k_recover_learned_vsq<MF, HB, HK, HEAT, 2>), g, wg, 0, s, L.k, F, S, W, R, A);
    else if (u == 1)
      hipLaunchKernelGGL((k_recover_learned_vsq<MF, HB, HK, HEAT, 1>), g, wg, 0, s, L.k, F, S, W, R, A);
    else
      hipLaunchKernelGGL((k_recover_learned_vsq<MF, HB, HK, HEAT, 0>), g, wg, 0, s, L.k, F, S, W, R, A);
  }
}

template <int MF, int REC, bool HB, bool HK, bool HEAT>
static void launch_queue(const LaunchCtx &L, const KFields &F, const SharedTabs &S, const Range3 &R, dim3 wg,
                         hipStream_t s) {
  const auto kernel = k_recover_queue<MF, REC, HB, HK, HEAT>;
  hipLaunchKernelGGL(kernel, dim3(resident_groups(kernel, R.tile, R.ntiles)), wg, 0, s, L.k, F, S, R, L.queue);
}

// W: the model's view, or null for the work queue.
template <int MF, bool HB, bool HK, bool HEAT>
static void launch_scheme(const LaunchCtx &L, const KFields &F, const SharedTabs &S, int rec, const MlpFrag *W,
                          const Range3 &R, dim3 g, dim3 wg, hipStream_t s, const UpdArgs *upd) {
  if (W)
    launch_learned<MF, HB, HK, HEAT>(L, F, S, *W, R, g, wg, s, upd);
  else if (rec == 0)
    launch_queue<MF, 0, HB, HK, HEAT>(L, F, S, R, wg, s);
  else if (rec == 1)
    launch_queue<MF, 1, HB, HK, HEAT>(L, F, S, R, wg, s);
  else if (rec == 2)
    launch_queue<MF, 2, HB, HK, HEAT>(L, F, S, R, wg, s);
  else if (HEAT)
    launch_queue<MF, -1, HB, HK, HEAT>(L, F, S, R, wg, s);
}
template <int MF, bool HB>
static void launch_fields(const LaunchCtx &L, const KFields &F, const SharedTabs &S, int rec, bool heat,
                          const MlpFrag *W, const Range3 &R, dim3 g, dim3 wg, hipStream_t s,
                          const UpdArgs *upd) {
  if (L.k.iKEL < 0)
    launch_scheme<MF, HB, false, false>(L, F, S, rec, W, R, g, wg, s, upd);
  else if (heat)
    launch_scheme<MF, HB, true, true>(L, F, S, rec, W, R, g, wg, s, upd);
  else
    launch_scheme<MF, HB, true, false>(L, F, S, rec, W, R, g, wg, s, upd);
}

void launch_recover_option(const LaunchCtx &L, const KFields &F, const SharedTabs &S, int rec, bool heat,
                           const MlpFrag *W, const Range3 &R, hipStream_t s, const UpdArgs *upd) {
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, nv = metric_form(L.metric) == FORM_NULLV;
  if (nv && hb)
    launch_fields<FORM_NULLV, true>(L, F, S, rec, heat, W, R, g, wg, s, upd);
  else if (nv)
    launch_fields<FORM_NULLV, false>(L, F, S, rec, heat, W, R, g, wg, s, upd);
  else if (hb)
    launch_fields<FORM_FULL, true>(L, F, S, rec, heat, W, R, g, wg, s, upd);
  else
    launch_fields<FORM_FULL, false>(L, F, S, rec, heat, W, R, g, wg, s, upd);
}

}  // namespace pangu
