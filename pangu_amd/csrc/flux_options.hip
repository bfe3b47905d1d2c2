// The other forms of the sweeps, which a run asks for: FixPrimitive and the X1
// sweep in one kernel, shared reconstruction, two lanes per face, marching
// columns.  (A file of their own: a program that never asks does not load
// them.)
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

// FixPrimitive + CalculateConservative (k_fix_cons) and the X1 sweep
// (k_flux<1>) in one pass.  A workgroup of 256 threads covers cells
// t0 - 4 .. t0 + R.tile + 3 of one ghosted plane (R: the entire range in runs
// of R.tile = 248 cells, decoded as decode_tile_at does), fixes every one of
// them and stores the outputs of the cells it owns (t0 .. t0 + 247); the
// four halo cells on each side are fixed again by the neighbouring
// workgroup (FixPrimitive is pointwise, so both compute the same bits).  The
// fixed primitives wait in LDS, and each owned cell that is an X1 face
// (s..e+1, one transverse ghost layer) reconstructs its two states from
// them: the stencil i-3..i+2 lies in the cell's row and in the window.  Same
// operations and operands as the two kernels: identical results.
template <int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256) void k_fix_flux_x1(KCtx C, KFields F, uint8_t *const *mask,
                                                     double *const *alfven, Range3 R) {
  __shared__ double sp[NPRIM][256];
  const int N = R.ntiles;
  const int n8 = (N + 7) >> 3;
  const int L = (int)blockIdx.x;
  const int T = (L & 7) * n8 + (L >> 3);
  if (T >= N) return;  // uniform over the workgroup
  const int TL = R.tile;
  int lo[3], cnt[3], local, tpp, b;
  if (R.uni) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = R.ulo[d];
      cnt[d] = R.ucnt[d];
    }
    tpp = R.utpp;
    const int per_block = cnt[2] * tpp;
    b = T / per_block;
    local = T - b * per_block;
  } else {
    b = R.tblock[T];
    local = T - R.tfirst[b];
    block_range(C.blk[b], R, lo, cnt);
    tpp = (cnt[0] * cnt[1] + TL - 1) / TL;
  }
  const int plane = cnt[0] * cnt[1];
  int tile, kk;
  if (R.order) {
    tile = local / cnt[2];
    kk = local - tile * cnt[2];
  } else {
    kk = local / tpp;
    tile = local - kk * tpp;
  }
  const int x = (int)threadIdx.x;
  const int t = tile * TL + x - 4;
  const bool valid = t >= 0 && t < plane && x < TL + 8;
  const bool own = valid && x >= 4 && x < TL + 4;
  const int k = lo[2] + kk;
  int j = 0, i = 0;
  if (valid) {
    const int jj = t / cnt[0];
    j = lo[1] + jj;
    i = lo[0] + (t - jj * cnt[0]);
  }
  double p[NPRIM];
#pragma unroll
  for (int q = 0; q < NPRIM; ++q) p[q] = 0.0;
  if (valid) fix_cons_cell<MF, true, true, HB, HK>(C, F, mask, b, k, j, i, own, p);
#pragma unroll
  for (int q = 0; q < NPRIM; ++q) sp[q][x] = p[q];
  __syncthreads();
  if (!own) return;
  const DevBlock &B = C.blk[b];
  const bool face = i >= B.s[0] && i <= B.e[0] + 1 &&
                    (B.n[1] > 1 ? (j >= B.s[1] - 1 && j <= B.e[1] + 1) : j == B.s[1]) &&
                    (B.n[2] > 1 ? (k >= B.s[2] - 1 && k <= B.e[2] + 1) : k == B.s[2]);
  if (!face) return;
  constexpr int NC = ncomp<HB, HK>();
  constexpr int NS = (LIM == PANGU_LIMITER_PPM4) ? 6 : 4;  // offsets -NS/2 .. NS/2 - 1
  double pl[NPRIM], pr[NPRIM];
#pragma unroll
  for (int q = 0; q < NPRIM; ++q) {
    pl[q] = 0.0;
    pr[q] = 0.0;
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int sl = slot_of<HB, HK>(q);
    double v[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) v[n] = sp[sl][x + n - NS / 2];
    double t0, t1;
    if (LIM == PANGU_LIMITER_PPM4) {
      recon_ppm4(v[0], v[1], v[2], v[3], v[4], pl[sl], t0);
      recon_ppm4(v[1], v[2], v[3], v[4], v[5], t1, pr[sl]);
    } else {
      recon_mc(v[0], v[1], v[2], pl[sl], t0);
      recon_mc(v[1], v[2], v[3], t1, pr[sl]);
    }
  }
  face_flux<1, RS, HB, HK, MF>(C, F, alfven, b, k, j, i, pl, pr);
}

// The value of lane l - 1 (lane 0 gets 0) through the DPP wavefront shift
// (wave_shr:1), 32 bits at a time.
__device__ __forceinline__ double wave_shr1(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x138, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// Exchange with the other lane of an aligned lane pair (l ^ 1) through the
// data-parallel-primitive path (quad_perm [1, 0, 3, 2]), 32 bits at a time.
__device__ __forceinline__ double pair_swap(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0xB1, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0xB1, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// Flux sweep with two lanes per face.  The even lane of a pair builds the
// left state (cell i - 1 along DIR), the odd lane the right state (cell i):
// each reconstructs one side (the stencil shared through the pair: each lane
// loads every other stencil cell and takes the rest from its partner), forms
// its fluid state, wave speeds and flux vectors, then the pair exchanges the
// speeds and the flux components the other lane combines; the even lane
// writes the first half of the components and the wave speed, the odd lane
// the rest.  Every value is computed by the same expressions in the same
// order as k_flux, so the results are identical; what changes is that one
// lane holds one fluid state instead of two (fewer registers, more
// wavefronts in flight).
template <int DIR, int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256) void k_flux_pair(KCtx C, KFields F, double *const *alfven, Range3 R) {
  int b = 0, k = 0, j = 0, i = 0;
  if (!decode_tile_pair(C, R, b, k, j, i)) return;  // both lanes of a pair share the outcome
  const int side = (int)threadIdx.x & 1;            // 0: left state, 1: right state
  const DevBlock &B = C.blk[b];
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t st = (DIR == 1) ? 1 : (DIR == 2 ? sj : sk);
  const int64_t id = k * sk + j * sj + i;
  constexpr int NC = ncomp<HB, HK>();
  constexpr int NS = (LIM == PANGU_LIMITER_PPM4) ? 6 : 4;  // stencil offsets -NS/2 .. NS/2 - 1
  constexpr int NL = NS / 2;                               // cells each lane loads
  double p[NPRIM];
#pragma unroll
  for (int q = 0; q < NPRIM; ++q) p[q] = 0.0;
  {
    // lane `side` loads offsets -NS/2 + side + 2m; its stencil for one side
    // is offsets side - NS/2 + n, n = 0 .. NS - 2
    double a[NC][NL];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const auto arr = glb(F.prim[b * NC + q]);
#pragma unroll
      for (int m = 0; m < NL; ++m) a[q][m] = arr[id + (2 * m + side - NS / 2) * st];
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      double x[NL], w[NS - 1];
#pragma unroll
      for (int m = 0; m < NL; ++m) x[m] = pair_swap(a[q][m]);
#pragma unroll
      for (int n = 0; n < NS - 1; ++n) {
        if ((n & 1) == 0)
          w[n] = a[q][n >> 1];
        else
          w[n] = side ? x[((n - 1) >> 1) + 1] : x[(n - 1) >> 1];
      }
      const int s = slot_of<HB, HK>(q);
      double t;
      if (LIM == PANGU_LIMITER_PPM4) {
        if (side == 0)
          recon_ppm4(w[0], w[1], w[2], w[3], w[4], p[s], t);
        else
          recon_ppm4(w[0], w[1], w[2], w[3], w[4], t, p[s]);
      } else {
        if (side == 0)
          recon_mc(w[0], w[1], w[2], p[s], t);
        else
          recon_mc(w[0], w[1], w[2], t, p[s]);
      }
    }
  }
  const DevGeo &G = C.geo[B.geo];
  double g[16], gc0[4], gdd, sg, alpha, valid;
  if (DIR == 3 && !G.face[2]) {
    const int64_t t = cen_index(G, k, j, i);
    const auto c = glb(G.cen);
    const int64_t ns = G.ncen;
    load_gcov([&](int n) { return c[n * ns + t]; }, MF == FORM_NULLV, g);
#pragma unroll
    for (int n = 0; n < 4; ++n) gc0[n] = c[(CG_GCON + n) * ns + t];
    gdd = c[(CG_GCON + 15) * ns + t];
    sg = c[CG_SG * ns + t];
    alpha = c[CG_ALPHA * ns + t];
    valid = 1.0;
  } else {
    const int d = DIR - 1;
    const int64_t t = ((int64_t)(G.has3d ? k : 0) * G.fj[d] + j) * G.fi[d] + i;
    const auto c = glb(G.face[d]);
    const int64_t ns = G.nface[d];
    load_gcov([&](int n) { return c[n * ns + t]; }, MF == FORM_NULLV, g);
#pragma unroll
    for (int n = 0; n < 4; ++n) gc0[n] = c[(FG_GCON0 + n) * ns + t];
    gdd = c[FG_GCONDD * ns + t];
    sg = c[FG_SG * ns + t];
    alpha = c[FG_ALPHA * ns + t];
    valid = c[FG_VALID * ns + t];
  }
  constexpr int NH = (NC + 1) / 2;  // components written by the even lane
  const auto al = glb(alfven[b * 3 + (DIR - 1)]);
  if (valid == 0.0) {  // the same for both lanes of the pair
    // singular face metric (polar axis): zero flux and wave speed
    if (side == 0) al[id] = 0.0;
#pragma unroll
    for (int q = 0; q < NC; ++q)
      if ((q < NH) == (side == 0)) glb(F.flux[DIR - 1][b * NC + q])[id] = 0.0;
    return;
  }
  const double gam = C.ph.gamma;
  St sm;
  calc_state(p, g, gc0, alpha, sm);
  double vmax, vmin;
  fast_ms<DIR>(gam, p, sm, gc0[0], gc0[DIR], gdd, vmax, vmin);
  const double vmaxO = pair_swap(vmax), vminO = pair_swap(vmin);
  const double vmaxL = side ? vmaxO : vmax, vminL = side ? vminO : vmin;
  const double vmaxR = side ? vmax : vmaxO, vminR = side ? vmin : vminO;
  const double cmax = fabs(kmax(kmax(0., vmaxL), vmaxR));
  const double cmin = fabs(kmax(kmax(0., -vminL), -vminR));
  const double cc = kmax(cmax, cmin);
  if (side == 0) al[id] = cc;
  double Um[NPRIM], Fm[NPRIM];
  contravariant_flux<0>(gam, p, sm, sg, Um);
  contravariant_flux<DIR>(gam, p, sm, sg, Fm);
  const double den = cmax + cmin + 1e-20, rden = 1.0 / den;
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int s = slot_of<HB, HK>(q);
    const double Uo = pair_swap(Um[s]), Fo = pair_swap(Fm[s]);
    if ((q < NH) == (side == 0)) {
      const double UL = side ? Uo : Um[s], UR = side ? Um[s] : Uo;
      const double FL = side ? Fo : Fm[s], FR = side ? Fm[s] : Fo;
      double f;
      if (RS == PANGU_RIEMANN_LAXF)
        f = 0.5 * (FL + FR - cc * (UR - UL));
      else
        f = div_by(cmax * FL + cmin * FR - cmax * cmin * (UR - UL), den, rden);
      glb(F.flux[DIR - 1][b * NC + q])[id] = f;
    }
  }
}

// X1 sweep with one reconstruction per cell.  Lane l of a wavefront
// reconstructs cell c (both interface values, the same PPM4 / MC call the
// face kernel makes) and takes the right interface value of cell c - 1 from
// lane l - 1, so each cell's reconstruction runs once instead of twice.
// Waves cover 64 consecutive cells of a plane's row-major cell range
// (i = s - 1 .. e + 1) and overlap by one cell, so both neighbours of every
// face sit in one wave.  Same arithmetic as k_flux<1>: identical results.
template <int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256) void k_flux_x1s(KCtx C, KFields F, double *const *alfven, Range3 R) {
  const int N = R.ntiles;
  const int n8 = (N + 7) >> 3;
  const int L = (int)blockIdx.x;
  const int T = (L & 7) * n8 + (L >> 3);
  if (T >= N) return;  // uniform over the workgroup
  const int b = R.tblock[T];
  const int local = T - R.tfirst[b];
  const DevBlock &B = C.blk[b];
  int lo[3], cnt[3];
  block_range(B, R, lo, cnt);
  const int plane = cnt[0] * cnt[1];
  const int wpp = (plane - 1 + 62) / 63;
  const int tpp = (wpp + 3) / 4;
  const int kk = local / tpp;
  const int w = (local - kk * tpp) * 4 + ((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const int cidx = w * 63 + lane;
  const bool have = (w < wpp) && (cidx < plane);
  const int jj = have ? cidx / cnt[0] : 0;
  const int ic = have ? cidx - jj * cnt[0] : 0;
  const int k = lo[2] + kk, j = lo[1] + jj, i = lo[0] + ic;
  const int64_t id = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  constexpr int NC = ncomp<HB, HK>();
  double rv[NPRIM], pl[NPRIM], pr[NPRIM];
#pragma unroll
  for (int s = 0; s < NPRIM; ++s) {
    rv[s] = 0.0;
    pl[s] = 0.0;
    pr[s] = 0.0;
  }
  // the cell stencils of every variable are loaded before the first
  // reconstruction (one wait for memory), then each cell's right interface
  // value moves one lane up through a DPP wavefront shift
  constexpr int NS = (LIM == PANGU_LIMITER_PPM4) ? 5 : 3;  // offsets -NS/2 .. NS/2
  double v[NC][NS];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const auto a = glb(F.prim[b * NC + q]);
#pragma unroll
    for (int n = 0; n < NS; ++n) v[q][n] = have ? a[id + (n - NS / 2)] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int s = slot_of<HB, HK>(q);
    if (LIM == PANGU_LIMITER_PPM4)
      recon_ppm4(v[q][0], v[q][1], v[q][2], v[q][3], v[q][4], rv[s], pr[s]);
    else
      recon_mc(v[q][0], v[q][1], v[q][2], rv[s], pr[s]);
    pl[s] = wave_shr1(rv[s]);
  }
  if (!have || lane == 0 || ic == 0) return;
  face_flux<1, RS, HB, HK, MF>(C, F, alfven, b, k, j, i, pl, pr);
}

// Marching sweep along DIR (2 or 3): each thread walks R.step consecutive
// faces of one column (decode_march) and reconstructs each cell of the
// column once.  Cell m's reconstruction gives the right state of face m
// and the left state of face m + 1; the latter waits in LDS (one slot per
// thread, read back by the same thread) while face m's physics runs, so
// the registers peak as in k_flux.  A column of s faces reconstructs s + 1
// cells instead of 2s.  Same inputs and arithmetic per face as k_flux:
// identical results.  On an MI355X it ran 15-35 % slower than k_flux on
// 64x64x32 blocks: a cell's reconstruction is only ~13 % of a face's FP64
// instructions, and each face's loads wait for the previous face's physics
// instead of overlapping other faces' work; the autotuner picks it only
// where it wins.
template <int DIR, int LIM, int RS, bool HB, bool HK, int MF>
__global__ __launch_bounds__(256, 3) void k_flux_march(KCtx C, KFields F, double *const *alfven,
                                                    Range3 R) {
  int b = 0, k = 0, j = 0, i = 0, mend = 0;
  if (!decode_march<DIR>(C, R, b, k, j, i, mend)) return;
  const DevBlock &B = C.blk[b];
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t st = (DIR == 2) ? sj : sk;
  constexpr int NC = ncomp<HB, HK>();
  constexpr int NS = (LIM == PANGU_LIMITER_PPM4) ? 5 : 3;  // offsets -NS/2 .. NS/2
  __shared__ double carry[NPRIM][TILE];
  const int tid = (int)threadIdx.x;
  double pl[NPRIM], pr[NPRIM];
#pragma unroll
  for (int s = 0; s < NPRIM; ++s) {
    pl[s] = 0.0;
    pr[s] = 0.0;
  }
  int &m = (DIR == 2) ? j : k;
  // the left state of the first face: cell m - 1 at its right face
  {
    const int64_t id = (int64_t)k * sk + (int64_t)j * sj + i - st;
    double v[NC][NS];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const auto a = glb(F.prim[b * NC + q]);
#pragma unroll
      for (int n = 0; n < NS; ++n) v[q][n] = a[id + (n - NS / 2) * st];
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int s = slot_of<HB, HK>(q);
      double t0;
      if (LIM == PANGU_LIMITER_PPM4)
        recon_ppm4(v[q][0], v[q][1], v[q][2], v[q][3], v[q][4], pl[s], t0);
      else
        recon_mc(v[q][0], v[q][1], v[q][2], pl[s], t0);
    }
  }
#pragma unroll 1
  for (; m < mend; ++m) {
    // an opaque step: every address below is formed from m afresh, so the
    // compiler keeps no per-array pointer alive across the iterations
    __asm__ volatile("" : "+v"(m));
    const int64_t id = (int64_t)k * sk + (int64_t)j * sj + i;
    double v[NC][NS];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const auto a = glb(F.prim[b * NC + q]);
#pragma unroll
      for (int n = 0; n < NS; ++n) v[q][n] = a[id + (n - NS / 2) * st];
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int s = slot_of<HB, HK>(q);
      double nx;
      if (LIM == PANGU_LIMITER_PPM4)
        recon_ppm4(v[q][0], v[q][1], v[q][2], v[q][3], v[q][4], nx, pr[s]);
      else
        recon_mc(v[q][0], v[q][1], v[q][2], nx, pr[s]);
      carry[s][tid] = nx;
    }
    // keep the carried states in LDS, not in registers, across the face
    // physics (the compiler would otherwise forward the stores)
    __asm__ volatile("" ::: "memory");
    face_flux<DIR, RS, HB, HK, MF>(C, F, alfven, b, k, j, i, pl, pr);
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int s = slot_of<HB, HK>(q);
      pl[s] = carry[s][tid];
    }
  }
}

// ===================================================================== host
template <int DIR>
static int sweep_option(const LaunchCtx &L, const KFields &F, double *const *alfven, hipStream_t s) {
  const bool shared = DIR == 1 && L.share_x1;
  constexpr int MD = DIR >= 2 ? DIR - 2 : 0;
  const bool march = DIR >= 2 && L.march_depth[MD] > 0;
  const bool pair = !shared && !march && ((L.pair_flux >> (DIR - 1)) & 1);
  if (!shared && !march && !pair) return 0;
  // these forms decode 256-cell tiles
  Range3 R = shared ? L.x1cells : march ? L.march[MD] : L.face[DIR - 1];
  R.order = L.order[PANGU_KF_FLUX_X1 + DIR - 1];
  if (R.ntiles == 0) return -1;
  const dim3 g = tile_grid(R);
  const dim3 g2((unsigned)(((2 * R.ntiles + 7) / 8) * 8));
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  const int lim = L.limiter, rs = L.riemann, mf = metric_form(L.metric);
#define FV(LIM, RS, HB_, HK_, MF_)                                                                 \
  if (shared)                                                                                     \
    hipLaunchKernelGGL((k_flux_x1s<LIM, RS, HB_, HK_, MF_>), g, kTile, 0, s, L.k, F, alfven, R);  \
  else if (march)                                                                                 \
    hipLaunchKernelGGL((k_flux_march<(DIR > 1 ? DIR : 2), LIM, RS, HB_, HK_, MF_>), g, kTile, 0, s, L.k, \
                       F, alfven, R);                                                             \
  else                                                                                            \
    hipLaunchKernelGGL((k_flux_pair<DIR, LIM, RS, HB_, HK_, MF_>), g2, kTile, 0, s, L.k, F, alfven, R)
#define FL(LIM, RS, HB_, HK_)                  \
  if (mf == FORM_NULLV) {                      \
    FV(LIM, RS, HB_, HK_, FORM_NULLV);         \
  } else {                                     \
    FV(LIM, RS, HB_, HK_, FORM_FULL);          \
  }
#define FL2(LIM, RS)                         \
  if (hb && hk) { FL(LIM, RS, true, true); } \
  else if (hb) { FL(LIM, RS, true, false); } \
  else if (hk) { FL(LIM, RS, false, true); } \
  else { FL(LIM, RS, false, false); }
  if (lim == PANGU_LIMITER_PPM4 && rs == PANGU_RIEMANN_LAXF) {
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
#undef FV
  return 1;
}

int launch_sweep_option(const LaunchCtx &L, int dir, const KFields &F, double *const *alfven, hipStream_t s) {
  return dir == 1 ? sweep_option<1>(L, F, alfven, s)
                  : dir == 2 ? sweep_option<2>(L, F, alfven, s) : sweep_option<3>(L, F, alfven, s);
}

template <int LIM, int RS, bool HB, bool HK>
static void launch_fx(const LaunchCtx &L, const Range3 &R, const KFields &F, uint8_t *const *mask,
                      double *const *alfven, hipStream_t s) {
  if (metric_form(L.metric) == FORM_NULLV)
    hipLaunchKernelGGL((k_fix_flux_x1<LIM, RS, HB, HK, FORM_NULLV>), tile_grid(R), kTile, 0, s, L.k, F, mask,
                       alfven, R);
  else
    hipLaunchKernelGGL((k_fix_flux_x1<LIM, RS, HB, HK, FORM_FULL>), tile_grid(R), kTile, 0, s, L.k, F, mask,
                       alfven, R);
}
template <int LIM, int RS>
static void launch_fx_fields(const LaunchCtx &L, const Range3 &R, const KFields &F, uint8_t *const *mask,
                             double *const *alfven, hipStream_t s) {
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  if (hb && hk)
    launch_fx<LIM, RS, true, true>(L, R, F, mask, alfven, s);
  else if (hb)
    launch_fx<LIM, RS, true, false>(L, R, F, mask, alfven, s);
  else if (hk)
    launch_fx<LIM, RS, false, true>(L, R, F, mask, alfven, s);
  else
    launch_fx<LIM, RS, false, false>(L, R, F, mask, alfven, s);
}

int launch_fix_flux_x1(const LaunchCtx &L, const KFields &F, uint8_t *const *mask, double *const *alfven,
                       hipStream_t s) {
  Range3 R = L.fixx1;
  R.order = L.order[PANGU_KF_FIX_CONS];
  if (R.ntiles == 0 || R.tile + 8 != TILE) return -1;
  if (L.limiter == PANGU_LIMITER_PPM4) {
    if (L.riemann == PANGU_RIEMANN_HLL)
      launch_fx_fields<PANGU_LIMITER_PPM4, PANGU_RIEMANN_HLL>(L, R, F, mask, alfven, s);
    else
      launch_fx_fields<PANGU_LIMITER_PPM4, PANGU_RIEMANN_LAXF>(L, R, F, mask, alfven, s);
  } else {
    if (L.riemann == PANGU_RIEMANN_HLL)
      launch_fx_fields<PANGU_LIMITER_MC, PANGU_RIEMANN_HLL>(L, R, F, mask, alfven, s);
    else
      launch_fx_fields<PANGU_LIMITER_MC, PANGU_RIEMANN_LAXF>(L, R, F, mask, alfven, s);
  }
  TICK("fix_cons_flux_x1");
  return PG_CHECK_LAUNCH();
}

}  // namespace pangu
