// gfx950 kernels of the GRMHD per-RK-stage update path (FP64 vector ALU).
//
// Thread mapping: a launch is a 1D grid of 256-thread tiles.  The (i, j)
// range of each (block, k) plane is flattened row-major, so consecutive lanes
// take consecutive i (coalesced loads) and rows of any width (65, 66, 72 ...)
// fill whole wavefronts.  All three flux sweeps therefore load coalesced
// rows; the reference's j- and k-innermost sweeps (laxf.cc:189,295) would
// stride through memory on a GPU.  Tiles are remapped so that consecutive
// logical tiles run on the same XCD: the hardware deals workgroups to the 8
// XCDs round-robin, and neighbouring tiles share stencil rows and planes
// through that XCD's L2.
#include <hip/hip_runtime.h>
#include <float.h>

#include "cell_dev.h"
#include "common.h"
#include "halo_dev.h"
#include "kernels.h"
#include "launch_host.h"
#include "physics_dev.h"
#include "recovery_dev.h"
#include "tiles_dev.h"
#include "update_dev.h"

namespace pangu {

// ------------------------------------------------------ constrained transport
// Corner EMFs (constrained_transport.cc:49-76).
__global__ __launch_bounds__(256) void k_emf(KCtx C, KFields F, double *const *emf, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  const DevBlock &B = C.blk[b];
  const bool o1 = B.n[0] > 1, o2 = B.n[1] > 1, o3 = B.n[2] > 1;
  const bool e1on = o2 && o3, e2on = o3 && o1, e3on = o1 && o2;
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t id = k * sk + j * sj + i;
  const int nc = C.nc;
  const int b1 = C.iBX, b2 = C.iBX + 1, b3 = C.iBX + 2;
  double e1 = 0.0, e2 = 0.0, e3 = 0.0;
  if (e1on) {
    const auto f2 = glb(F.flux[1][b * nc + b3]), f3 = glb(F.flux[2][b * nc + b2]);
    e1 = 0.25 * ((f2[id] + f2[id - sk]) - (f3[id] + f3[id - sj]));
  }
  if (e2on) {
    const auto f3 = glb(F.flux[2][b * nc + b1]), f1 = glb(F.flux[0][b * nc + b3]);
    e2 = 0.25 * ((f3[id] + f3[id - 1]) - (f1[id] + f1[id - sk]));
  }
  if (e3on) {
    const auto f1 = glb(F.flux[0][b * nc + b2]), f2 = glb(F.flux[1][b * nc + b1]);
    e3 = 0.25 * ((f1[id] + f1[id - sj]) - (f2[id] + f2[id - 1]));
  }
  glb(emf[b * 3 + 0])[id] = e1;
  glb(emf[b * 3 + 1])[id] = e2;
  glb(emf[b * 3 + 2])[id] = e3;
}

// Face B-flux overwrite from the EMFs (constrained_transport.cc:78-127).
// One launch covers the union of the three face ranges.
__global__ __launch_bounds__(256) void k_ct_faces(KCtx C, KFields F, double *const *emf, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  const DevBlock &B = C.blk[b];
  const int o1 = B.n[0] > 1, o2 = B.n[1] > 1, o3 = B.n[2] > 1;
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t id = k * sk + j * sj + i;
  const int nc = C.nc;
  const int b1 = C.iBX, b2 = C.iBX + 1, b3 = C.iBX + 2;
  const int E1 = o2 && o3, E2 = o3 && o1, E3 = o1 && o2;
  const auto e1 = glb(emf[b * 3 + 0]), e2 = glb(emf[b * 3 + 1]), e3 = glb(emf[b * 3 + 2]);
  const bool in_k = k <= B.e[2], in_j = j <= B.e[1], in_i = i <= B.e[0];
  if (in_k && in_j) {  // X1 faces: i in [is, ie+o1]
    if (o1) glb(F.flux[0][b * nc + b1])[id] = 0;
    if (E2) glb(F.flux[0][b * nc + b3])[id] = -0.5 * (e2[id] + e2[id + sk]);
    if (E3) glb(F.flux[0][b * nc + b2])[id] = 0.5 * (e3[id] + e3[id + sj]);
  }
  if (in_k && in_i) {  // X2 faces: j in [js, je+o2]
    if (E1) glb(F.flux[1][b * nc + b3])[id] = 0.5 * (e1[id] + e1[id + sk]);
    if (o2) glb(F.flux[1][b * nc + b2])[id] = 0.;
    if (E3) glb(F.flux[1][b * nc + b1])[id] = -0.5 * (e3[id] + e3[id + 1]);
  }
  if (in_j && in_i && o3) {  // X3 faces: k in [ks, ke+o3]
    if (E1) glb(F.flux[2][b * nc + b2])[id] = -0.5 * (e1[id] + e1[id + sj]);
    if (E2) glb(F.flux[2][b * nc + b1])[id] = 0.5 * (e2[id] + e2[id + 1]);
    glb(F.flux[2][b * nc + b3])[id] = 0;
  }
}

template <int MODE, int MF, bool HB, bool HK, bool CTF>
__global__ __launch_bounds__(256, (HB && MODE != 1) ? 5 : 4) void k_div_update(KCtx C, KFields F0, KFields Finit, KFields F1,
                                                    double *const *dudt,
                                                    const double *dt_dev, double beta,
                                                    double bdt_host, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  div_update_cell<MODE, MF, HB, HK, CTF>(C, F0, Finit, F1, dudt, dt_dev, beta, bdt_host, b, k, j, i,
                                          nullptr);
}

template <int MF, int REC, bool HB, bool HK, bool HEAT>
__global__ __launch_bounds__(256) void k_recover(KCtx C, KFields F, SharedTabs S, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  recover_cell<MF, REC, HB, HK, HEAT>(C, F, S, b, k, j, i);
}

// The update of k_div_update (mode 4: flux divergence, RK update, source)
// and the recovery (+ heating) of k_recover for the same cell in one pass:
// the recovery takes the new U from registers instead of memory.  The update
// is memory-bound and the recovery VALU-bound, so their phases overlap
// across the wavefronts of one launch.  Same operations per cell in the same
// order: identical results.  Called only when nothing has to run between
// the two (the stage's exchange runs before).
// The metric's form (physics_dev.h) keeps what no cell of a mesh needs out of
// the registers: MKS with Kastaun and heating 165 -> 127 VGPRs (four
// wavefronts per SIMD instead of three) and 309 -> 288 loads; per cycle
// 4.186 -> 4.158 ms on the 3-D torus 256x128x128, 233 -> 227 us on the 2-D
// torus 512x256, 118 -> 109 us on Orszag-Tang 256^2; the chainer alone on a
// flat 301x199 plane 15.2 -> 11.0 us.
template <int MF, bool HB, bool HK, bool CTF, int REC, bool HEAT>
__global__ __launch_bounds__(256) void k_update_recover(KCtx C, KFields F0, KFields Finit, KFields F1,
                                                        SharedTabs S, const double *dt_dev, double beta,
                                                        double bdt_host, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  double u[NPRIM];
  div_update_cell<4, MF, HB, HK, CTF>(C, F0, Finit, F1, nullptr, dt_dev, beta, bdt_host, b, k, j, i, u);
  recover_cell<MF, REC, HB, HK, HEAT>(C, F1, S, b, k, j, i, -1.0, u);
}

// ---------------------------------------------------------- FixRecovery
// recovery_fixer.cc:216-285 with the serial (lexicographic, in-place)
// semantics of a single-threaded host build.  Phase A fixes failed cells
// with no failed 8-neighbour in parallel (nobody else reads or writes their
// stencils); cells touching another failed cell are left for phase B,
// which fixes each (block, k) plane's in an order equivalent to the
// lexicographic one.
//
// u~ becomes zero, every other component the mean over neighbours: the four
// nearest if all of them are good, else the four diagonal ones if all of
// those are, else all eight.  All values are loaded before the first store
// (which may alias them, as far as the compiler knows).
template <int NP>
__device__ __forceinline__ void fix_cell(double *const *pp, int64_t id, int64_t jp, const double *fl) {
  const int pf1 = (int)fl[id + jp - 1], pf2 = (int)fl[id + jp], pf3 = (int)fl[id + jp + 1];
  const int pf4 = (int)fl[id + 1];
  const int pf5 = (int)fl[id - jp + 1], pf6 = (int)fl[id - jp], pf7 = (int)fl[id - jp - 1];
  const int pf8 = (int)fl[id - 1];
  double *a[NP];
  double v[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    a[q] = pp[q];
    v[q] = 0.;
  }
  if (pf2 && pf4 && pf6 && pf8) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
      if (q < 2 || q > 4) v[q] = 0.25 * (glb(a[q])[id + jp] + glb(a[q])[id - jp] + glb(a[q])[id - 1] + glb(a[q])[id + 1]);
  } else if (pf1 && pf3 && pf5 && pf7) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
      if (q < 2 || q > 4)
        v[q] = 0.25 * (glb(a[q])[id + jp + 1] + glb(a[q])[id + jp - 1] + glb(a[q])[id - jp + 1] +
                       glb(a[q])[id - jp - 1]);
  } else {
#pragma unroll
    for (int q = 0; q < NP; ++q)
      if (q < 2 || q > 4)
        v[q] = 0.125 * (glb(a[q])[id + jp - 1] + glb(a[q])[id + jp] + glb(a[q])[id + jp + 1] + glb(a[q])[id + 1] +
                        glb(a[q])[id - jp + 1] + glb(a[q])[id - jp] + glb(a[q])[id - jp - 1] + glb(a[q])[id - 1]);
  }
#pragma unroll
  for (int q = 0; q < NP; ++q) glb(a[q])[id] = v[q];
}

// Is cell (k, j, i) excised?
__device__ __forceinline__ bool excised_cell(const KCtx &C, const DevBlock &B, int k, int j, int i) {
  if (C.ph.metric != PANGU_METRIC_CKS) return false;
  const DevGeo &G = C.geo[B.geo];
  return G.cen[CG_RAD * G.ncen + cen_index(G, k, j, i)] < C.ph.r_excise;
}

template <int NP>
__global__ __launch_bounds__(256) void k_fixrec_a(KCtx C, KFields F, double *const *flag,
                                                  int *cluster, Range3 R) {
  int b, k, j, i;
  if (!decode_tile(C, R, b, k, j, i)) return;
  const DevBlock &B = C.blk[b];
  const int64_t id = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  double *fl = flag[b];
  if (fl[id] != 0 || excised_cell(C, B, k, j, i)) return;
  const int64_t jp = (B.s[1] != B.e[1]) ? (int64_t)B.n[0] : 0;
  const bool isolated = fl[id + jp - 1] != 0 && fl[id + jp] != 0 && fl[id + jp + 1] != 0 &&
                        fl[id + 1] != 0 && fl[id - jp + 1] != 0 && fl[id - jp] != 0 &&
                        fl[id - jp - 1] != 0 && fl[id - 1] != 0;
  if (!isolated) {
    atomicOr(&cluster[C.pfirst[b] + k - B.s[2]], 1);
    return;
  }
  fix_cell<NP>(F.prim + b * NP, id, jp, fl);
  fl[id] = 1;
}

// Phase B: one wavefront per interior (block, k) plane that holds clustered
// cells (workgroup index = plane index).  Lane r walks row r of a band of 64
// rows, two columns behind lane r - 1: cell (r, c) is fixed in step c + 2 r.
// When a cell's turn comes, its neighbours to the left and in the row before
// are done and those to the right and in the row after are untouched, as in
// the lexicographic order, and no lane reads what another writes in the same
// step.  The failed cells are looked up first, as one bit per row in a word
// per step, and only steps with a bit set are taken (a cell's failure ends in
// its own turn and no other): a step is two memory round trips long, and of a
// band's ni + 126 steps a few clusters leave most empty.  The words of
// kFixSteps steps are held at a time.
// us per plane with        1 pair, 4 and 32 pairs of failed cells, all failed
//   64x64   as it is          11     16     55      205
//           every step taken  44     60     94      241
//           cell by cell      32     47    186    11400
//   512x256 as it is         237    242    285     4280
//           every step taken 640    699   1058     5110
//           cell by cell     686    701    833   375000
// (cell by cell: one lane, rows in turn).  First cycle of a 512x256 torus,
// whose atmosphere fails by the thousand: 5.0, 5.6 and 90 ms.
constexpr int kFixSteps = 1024;

template <int NP>
__global__ __launch_bounds__(64) void k_fixrec_b(KCtx C, KFields F, double *const *flag,
                                                 int *cluster) {
  __shared__ unsigned long long todo[kFixSteps];  // bit r: row r has a failed cell in this step
  const int b = C.pblock[blockIdx.x];
  const int kk = (int)blockIdx.x - C.pfirst[b];
  if (cluster[blockIdx.x] == 0) return;
  const DevBlock &B = C.blk[b];
  const int k = B.s[2] + kk;
  const int64_t jp = (B.s[1] != B.e[1]) ? (int64_t)B.n[0] : 0;
  double *fl = flag[b];
  const int lane = threadIdx.x;
  const int ni = B.e[0] - B.s[0] + 1;
  for (int j0 = B.s[1]; j0 <= B.e[1]; j0 += 64) {
    const int rows = min(64, B.e[1] - j0 + 1), steps = ni + 2 * (rows - 1);
    const int64_t row0 = ((int64_t)k * B.n[1] + j0) * B.n[0] + B.s[0];
    for (int s0 = 0; s0 < steps; s0 += kFixSteps) {
      const int ns = min(kFixSteps, steps - s0);
      for (int t = lane; t < ns; t += 64) todo[t] = 0ull;
      __syncthreads();
      // the columns that any row reaches in these steps
      const int c0 = max(0, s0 - 2 * (rows - 1)), nc = min(ni, s0 + ns) - c0, cells = rows * nc;
      for (int t = lane; t < cells; t += 64 * 8) {
        double f[8];
        int r[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int q = min(t + 64 * u, cells - 1);
          r[u] = q / nc;
          c[u] = c0 + q - r[u] * nc;
          f[u] = glb(fl)[row0 + (int64_t)r[u] * B.n[0] + c[u]];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int s = c[u] + 2 * r[u] - s0;
          if (f[u] == 0 && s >= 0 && s < ns && !excised_cell(C, B, k, j0 + r[u], B.s[0] + c[u]))
            atomicOr(&todo[s], 1ull << r[u]);
        }
      }
      __syncthreads();
      for (int t = 0; t < ns; t += 64) {
        const unsigned long long mine = t + lane < ns ? todo[t + lane] : 0ull;
        uint64_t left = __ballot(mine != 0);
        while (left) {
          const int l = __ffsll((unsigned long long)left) - 1;
          left &= left - 1;
          if ((__shfl(mine, l, 64) >> lane) & 1) {
            const int64_t id = row0 + (int64_t)lane * B.n[0] + (s0 + t + l - 2 * lane);
            fix_cell<NP>(F.prim + b * NP, id, jp, fl);
            fl[id] = 1;
          }
          __threadfence_block();  // the next step of every lane sees this one's stores
        }
      }
      __syncthreads();
    }
  }
  if (lane == 0) cluster[blockIdx.x] = 0;
}

// ------------------------------------------------- ghost exchange and BCs
// One thread per ghost cell.
template <int NP>
__global__ __launch_bounds__(256) void k_exchange(KCtx C, KFields F, double *const *flag,
                                                  const int *nbr, Items I) {
  int b, g;
  decode_item(I, b, g);
  exchange_cell<NP>(C, F, flag, nbr, b, g);
}

// Cell g of the two ghost slabs normal to d (side 0 below s[d], side 1 above
// e[d]), each ng layers deep and spanning the full ghosted extent of the
// other dims; i is fastest except for d = 0, where the layer index is.
__device__ __forceinline__ void bc_cell(const DevBlock &B, int d, int g, int &side, int &k, int &j,
                                        int &i) {
  const int ng = B.s[d];
  int ix[3];
  if (d == 0) {
    const int na = B.n[1], nb = B.n[2], per = ng * na * nb;
    side = g / per;
    const int r = g - side * per, kk = r / (na * ng), r2 = r - kk * na * ng, jj = r2 / ng;
    ix[0] = r2 - jj * ng;
    ix[1] = jj;
    ix[2] = kk;
  } else if (d == 1) {
    const int na = B.n[0], nb = B.n[2], per = ng * na * nb;
    side = g / per;
    const int r = g - side * per, kk = r / (ng * na), r2 = r - kk * ng * na, l = r2 / na;
    ix[0] = r2 - l * na;
    ix[1] = l;
    ix[2] = kk;
  } else {
    const int na = B.n[0], nb = B.n[1], per = ng * na * nb;
    side = g / per;
    const int r = g - side * per, l = r / (nb * na), r2 = r - l * nb * na, jj = r2 / na;
    ix[0] = r2 - jj * na;
    ix[1] = jj;
    ix[2] = l;
  }
  if (side == 1) ix[d] = B.e[d] + 1 + ix[d];
  i = ix[0];
  j = ix[1];
  k = ix[2];
}

// Physical boundaries: outflow copies the edge cell; reflecting mirrors and
// flips the d-component of u~ and B.  Semantics of the X1, X2 and X3 passes
// run in turn, each over the full extent of the other dims (so that corners
// fill from ghosts the earlier pass wrote).  Here each ghost cell takes the
// composition of those maps: the cell is carried back through X3, X2 and X1
// wherever it lies beyond a physical face, to a cell that no pass writes, so
// one launch serves all three.  One thread per cell of the two ghost slabs of
// every dim of a block that has a physical face; a cell beyond physical
// faces of several dims belongs to the slab of the highest.
template <int NP>
__global__ __launch_bounds__(256) void k_bc(KCtx C, KFields F, double *const *flag, Items I) {
  int b, g;
  decode_item(I, b, g);
  const DevBlock &B = C.blk[b];
  int d = 0;
  bool in = false;
  for (; d < 3; ++d) {
    if (B.bcf[d][0] < 0 && B.bcf[d][1] < 0) continue;
    const int slab = 2 * B.s[d] * (d == 0 ? B.n[1] * B.n[2] : (d == 1 ? B.n[0] * B.n[2] : B.n[0] * B.n[1]));
    in = g < slab;
    if (in) break;
    g -= slab;
  }
  if (!in) return;
  int side, k, j, i;
  bc_cell(B, d, g, side, k, j, i);
  if (B.bcf[d][side] < 0) return;
  const int ix[3] = {i, j, k};
  int sx[3] = {i, j, k};
  unsigned flip = 0;
  const int iBX = C.iBX;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    if (ix[e] >= B.s[e] && ix[e] <= B.e[e]) continue;
    const int kind = B.bcf[e][ix[e] < B.s[e] ? 0 : 1];
    if (kind < 0) continue;
    if (e > d) return;  // the slab of the higher dim covers this cell
    if (kind == PANGU_BC_OUTFLOW) {
      sx[e] = ix[e] < B.s[e] ? B.s[e] : B.e[e];
    } else {
      sx[e] = ix[e] < B.s[e] ? (2 * B.s[e] - 1 - ix[e]) : (2 * B.e[e] + 1 - ix[e]);
      flip |= 1u << (2 + e);
      if (iBX >= 0) flip |= 1u << (iBX + e);
    }
  }
  const int64_t dst = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  const int64_t src = ((int64_t)sx[2] * B.n[1] + sx[1]) * B.n[0] + sx[0];
  copy_cell<NP>(F, flag, b, dst, b, src, flip);
}

// --------------------------------------------------------------- timestep
// Per block and active direction the maximum face speed over interior
// cells; min_cells(cfl dx / c) equals cfl dx / max_cells(c) because IEEE
// division is monotone.  NaN speeds are skipped, as the reference's
// `if (dt_min > dt)` reduction skips NaN.  One workgroup per item (block,
// interior plane, chunk of 256 * PER cells of the plane) writes its maxima
// to red[item*3 + d]; no atomics, so the result is deterministic.
template <int PER>
__global__ __launch_bounds__(256) void k_dt_reduce(KCtx C, double *const *alfven, double *red) {
  __shared__ double sm[4][3];
  // thread x takes cells x, x + 256, ... of the chunk, all loads in flight
  // together (the maximum does not depend on the order)
  constexpr int kPer = PER, kDtChunk = 256 * PER;
  const int b = C.dtblock[blockIdx.x];
  const int local = (int)blockIdx.x - C.dtfirst[b];
  const DevBlock &B = C.blk[b];
  const int ni = B.e[0] - B.s[0] + 1, nj = B.e[1] - B.s[1] + 1;
  const int nch = (ni * nj + kDtChunk - 1) / kDtChunk;
  const int kk = local / nch, ch = local - kk * nch;
  const int k = B.s[2] + kk;
  const int t0 = ch * kDtChunk, t1 = (t0 + kDtChunk < ni * nj) ? t0 + kDtChunk : ni * nj;
  // (j, i) of cell t, stepped by 256 cells without a division per step
  const int dj = 256 / ni, di = 256 - dj * ni;
  int t = t0 + (int)threadIdx.x;
  int j = t / ni, i = t - j * ni;
  // steps holding a cell for some thread (the same for the whole workgroup:
  // a small plane skips the rest)
  const int nr = (t1 - t0 + 255) / 256;
  double v[kPer][3];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int64_t id = ((int64_t)k * B.n[1] + (B.s[1] + j)) * B.n[0] + (B.s[0] + i);
#pragma unroll
    for (int d = 0; d < 3; ++d)
      v[r][d] = (r < nr && t < t1 && B.n[d] != 1) ? glb(alfven[b * 3 + d])[id] : 0.0;
    t += 256;
    i += di;
    j += dj;
    if (i >= ni) {
      i -= ni;
      ++j;
    }
  }
  double c[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < kPer; ++r)
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (v[r][d] > c[d]) c[d] = v[r][d];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int d = 0; d < 3; ++d) {
    double v = c[d];
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(v, off, 64);
      v = (o > v) ? o : v;
    }
    if (lane == 0) sm[w][d] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int d = threadIdx.x;
    double v = sm[0][d];
    for (int q = 1; q < 4; ++q) v = (sm[q][d] > v) ? sm[q][d] : v;
    red[(int64_t)blockIdx.x * 3 + d] = v;
  }
}

// Harmonic combination per block (timestep_estimation.cc:94-98), minimum
// over the blocks of one mesh, then dt control dt_next = min(dt_factor * dt,
// estimate) and time += dt.  One workgroup per mesh m: state + 2m = {dt,
// time}; est_out (optional) + m gets the estimate.  W lanes share a block's
// items, which the maximum lets them read in any order: the kernel is a few
// memory round trips long, one for every 1024 / W blocks and one for every 4 W
// items of a block, and W is chosen for the fewest (LaunchCtx::dtlanes).  With
// 16 lanes for every mesh of more than 16 blocks, 512 blocks of 8^3 cells took
// 23.3 us, 1024 of 8^2 40.7 us and 2000 one-dimensional ones 68 us; with 2, 1
// and 1 lanes 6.9, 5.4 and 9.2 us; one block of 256^2 cells 4.0 us (64 lanes).
template <int W>
__global__ __launch_bounds__(1024) void k_dt_final(KCtx C, const double *red, double *state,
                                                   double dt_factor, double *est_out) {
  __shared__ double sm[16];
  const int m = blockIdx.x;
  const int lane = (int)threadIdx.x & (W - 1), grp = (int)threadIdx.x / W;
  double mn = DBL_MAX;
  for (int b = C.mfirst[m] + grp; b < C.mfirst[m + 1]; b += 1024 / W) {
    const DevBlock &B = C.blk[b];
    const int p1 = C.dtfirst[b + 1];
    double cmax[3] = {0.0, 0.0, 0.0};
    for (int p = C.dtfirst[b] + lane; p < p1; p += 4 * W) {
      double w[4][3];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int d = 0; d < 3; ++d) w[u][d] = (p + u * W < p1) ? red[(int64_t)(p + u * W) * 3 + d] : 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int d = 0; d < 3; ++d) cmax[d] = (w[u][d] > cmax[d]) ? w[u][d] : cmax[d];
    }
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double o = __shfl_xor(cmax[d], off, W);
        cmax[d] = (o > cmax[d]) ? o : cmax[d];
      }
    double q3[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (B.n[d] == 1) continue;
      const double q = C.ph.cfl * B.dx[d] / cmax[d];
      q3[d] = (q < DBL_MAX) ? q : DBL_MAX;
    }
    const double t = 1.0 / (1.0 / q3[0] + 1.0 / q3[1] + 1.0 / q3[2]);
    if (t < mn) mn = t;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(mn, off, 64);
    if (o < mn) mn = o;
  }
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = mn;
  __syncthreads();
  if (threadIdx.x == 0) {
    double est = sm[0];
    for (int q = 1; q < 16; ++q) est = (sm[q] < est) ? sm[q] : est;
    if (est_out) est_out[m] = est;
    if (state) {
      double *st = state + 2 * m;
      const double dt = st[0];
      st[1] = st[1] + dt;
      const double grown = dt_factor * dt;
      st[0] = (est < grown) ? est : grown;
    }
  }
}

// ===================================================================== host
hipError_t KernelClock::mark(const char *name, hipStream_t s) {
  if (n == events.size()) {
    hipEvent_t e;
    const hipError_t r = hipEventCreate(&e);
    if (r != hipSuccess) return r;
    events.push_back(e);
  }
  if (n > 0) {
    if (names.size() < n) names.resize(n);
    names[n - 1] = name;
  }
  return hipEventRecord(events[n++], s);
}

KernelClock::~KernelClock() {
  for (hipEvent_t e : events) (void)hipEventDestroy(e);
}

int launch_ct(const LaunchCtx &L, const KFields &F, double *const *emf, hipStream_t s) {
  const Range3 R = family_range(L, 5, L.ct, PANGU_KF_CT);
  if (R.ntiles == 0) return 0;
  const dim3 g = tile_grid(R), wg(R.tile);
  hipLaunchKernelGGL(k_emf, g, wg, 0, s, L.k, F, emf, R);
  TICK("ct_emf");
  hipLaunchKernelGGL(k_ct_faces, g, wg, 0, s, L.k, F, emf, R);
  TICK("ct_faces");
  return PG_CHECK_LAUNCH();
}

int launch_div_update(const LaunchCtx &L, int mode, const KFields &F0, const KFields &Finit,
                      const KFields &F1, double *const *dudt, bool ct_fused,
                      const double *dt_dev, double beta, double bdt_host, hipStream_t s) {
  const Range3 R = family_range(L, 0, L.interior, PANGU_KF_DIV_UPDATE);
  if (R.ntiles == 0) return 0;
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  const bool src = L.metric != PANGU_METRIC_MINKOWSKI;
  // CT fused into the divergence (modes 4 and 5 with a field)
  const bool ctf = ct_fused && hb && (mode == 4 || mode == 5);
#define DU(M, MF_, HB_, HK_, CT_)                                                               \
  hipLaunchKernelGGL((k_div_update<M, MF_, HB_, HK_, CT_>), g, wg, 0, s, L.k, F0, Finit, F1, \
                     dudt, dt_dev, beta, bdt_host, R)
#define DU2(M, MF_)                                      \
  if (hb && hk) {                                        \
    if ((M) == 4 && ctf) DU(M, MF_, true, true, (M) == 4); \
    else DU(M, MF_, true, true, false);                  \
  } else if (hb) {                                       \
    if ((M) == 4 && ctf) DU(M, MF_, true, false, (M) == 4); \
    else DU(M, MF_, true, false, false);                 \
  } else if (hk) DU(M, MF_, false, true, false);         \
  else DU(M, MF_, false, false, false);
  const int mf = metric_form(L.metric);  // FORM_FLAT: no source term
  switch (mode) {
    case 1: DU2(1, FORM_FLAT) break;
    case 2: DU2(2, FORM_FLAT) break;
    case 3:
      if (mf == FORM_POLOIDAL) {
        DU2(3, FORM_POLOIDAL)
      } else if (mf == FORM_NULLV) {
        DU2(3, FORM_NULLV)
      }
      break;
    case 5: DU2(4, FORM_FLAT) break;
    default:
      if (mf == FORM_POLOIDAL) {
        DU2(4, FORM_POLOIDAL)
      } else if (mf == FORM_NULLV) {
        DU2(4, FORM_NULLV)
      } else {
        DU2(4, FORM_FLAT)
      }
  }
#undef DU2
#undef DU
  if (mode != 3 || src)
    TICK(mode == 1   ? "flux_divergence"
         : mode == 2 ? "update"
         : mode == 3 ? "source"
         : mode == 5 ? "div_update"
                     : "div_update_source");
  return PG_CHECK_LAUNCH();
}

int launch_recover(const LaunchCtx &L, const KFields &F, const SharedTabs &S, int rec, bool heat,
                   const MlpFrag *W, hipStream_t s, const UpdArgs *upd) {
  // a fused update needs the learned kernel of the scheme (k_update_recover
  // serves the plain ones) and the range of the update
  if (upd && !(W && ((rec == 1 && W->kind == 0) || (rec == 2 && W->kind == 1)))) return -1;
  const Range3 R = upd ? family_range(L, 0, L.interior, PANGU_KF_DIV_UPDATE)
                       : family_range(L, 0, L.interior, PANGU_KF_RECOVERY);
  if (R.ntiles == 0) return 0;
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0;
  const bool persist = L.persist_recovery && L.queue;
  const int mf = metric_form(L.metric);
#define RC(R_, HB_, HK_, HE_)                                                                        \
  if (mf == FORM_POLOIDAL)                                                                            \
    hipLaunchKernelGGL((k_recover<FORM_POLOIDAL, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R);     \
  else if (mf == FORM_FLAT)                                                                           \
    hipLaunchKernelGGL((k_recover<FORM_FLAT, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R);         \
  else                                                                                                \
    hipLaunchKernelGGL((k_recover<FORM_NULLV, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R)
// (heating comes with K_e)
#define RC2(R_)                                  \
  if (hb && h) { RC(R_, true, true, true); }     \
  else if (h) { RC(R_, false, true, true); }     \
  else if (hb && hk) { RC(R_, true, true, false); } \
  else if (hb) { RC(R_, true, false, false); }   \
  else if (hk) { RC(R_, false, true, false); }   \
  else { RC(R_, false, false, false); }
  const bool h = heat && hk;
  const bool learned = W && ((rec == 1 && W->kind == 0) || (rec == 2 && W->kind == 1));
  if (learned || persist) {
    launch_recover_option(L, F, S, rec, h, learned ? W : nullptr, R, s, upd);
  } else if (rec == 0) {
    RC2(0)
  } else if (rec == 1) {
    RC2(1)
  } else if (rec == 2) {
    RC2(2)
  } else if (h && hb) {
    RC(-1, true, true, true);
  } else if (h) {
    RC(-1, false, true, true);
  }
#undef RC2
#undef RC
  if (rec >= 0 || h) TICK(rec < 0 ? "heating" : h ? "recovery_heating" : "recovery");
  return PG_CHECK_LAUNCH();
}

// Arguments of one k_update_recover launch, and the dispatch over its
// compile-time options: field (with CT formed in the update), K_e, heating
// and the recovery scheme.
struct URArgs {
  const KCtx &k;
  const KFields &F0, &Finit, &F1;
  const SharedTabs &S;
  const double *dt_dev;
  double beta, bdt_host;
  const Range3 &R;
};
template <int MF, bool HB, bool HK, int REC, bool HEAT>
static void launch_ur(const URArgs &a, dim3 g, dim3 wg, hipStream_t s) {
  hipLaunchKernelGGL((k_update_recover<MF, HB, HK, HB, REC, HEAT>), g, wg, 0, s, a.k, a.F0, a.Finit,
                     a.F1, a.S, a.dt_dev, a.beta, a.bdt_host, a.R);
}
template <int MF, int REC>
static void launch_ur_fields(const URArgs &a, dim3 g, dim3 wg, hipStream_t s, bool hb, bool hk, bool h) {
  if (!hb)
    launch_ur<MF, false, false, REC, false>(a, g, wg, s);
  else if (h)
    launch_ur<MF, true, true, REC, true>(a, g, wg, s);
  else if (hk)
    launch_ur<MF, true, true, REC, false>(a, g, wg, s);
  else
    launch_ur<MF, true, false, REC, false>(a, g, wg, s);
}
template <int MF>
static void launch_ur_rec(const URArgs &a, dim3 g, dim3 wg, hipStream_t s, int rec, bool hb, bool hk,
                          bool h) {
  if (rec == 0)
    launch_ur_fields<MF, 0>(a, g, wg, s, hb, hk, h);
  else if (rec == 1)
    launch_ur_fields<MF, 1>(a, g, wg, s, hb, hk, h);
  else
    launch_ur_fields<MF, 2>(a, g, wg, s, hb, hk, h);
}

int launch_update_recover(const LaunchCtx &L, const KFields &F0, const KFields &Finit,
                          const KFields &F1, const SharedTabs &S, int rec, bool heat, bool ct_fused,
                          const double *dt_dev, double beta, double bdt_host, hipStream_t s) {
  const Range3 R = family_range(L, 0, L.interior, PANGU_KF_DIV_UPDATE);
  if (R.ntiles == 0) return 0;
  const dim3 g = tile_grid(R), wg(R.tile);
  const bool hb = L.k.iBX >= 0, hk = L.k.iKEL >= 0, h = heat && hk;
  if ((hb && !ct_fused) || (!hb && hk) || rec < 0 || rec > 2) return -1;
  const URArgs a{L.k, F0, Finit, F1, S, dt_dev, beta, bdt_host, R};
  const int mf = metric_form(L.metric);
  if (mf == FORM_POLOIDAL)
    launch_ur_rec<FORM_POLOIDAL>(a, g, wg, s, rec, hb, hk, h);
  else if (mf == FORM_FLAT)
    launch_ur_rec<FORM_FLAT>(a, g, wg, s, rec, hb, hk, h);
  else
    launch_ur_rec<FORM_NULLV>(a, g, wg, s, rec, hb, hk, h);
  TICK("update_recovery");
  return PG_CHECK_LAUNCH();
}

// f<NP>() for the context's packed component count: 6, and 3 more with a
// field, 1 more with K_e.
#define WITH_NP(np, CALL) \
  switch (np) {           \
    case 6: CALL(6); break;   \
    case 7: CALL(7); break;   \
    case 9: CALL(9); break;   \
    default: CALL(10); break; \
  }

int launch_fix_recovery(const LaunchCtx &L, const KFields &F, double *const *flag, int *cluster,
                        hipStream_t s) {
  const Range3 &R = L.interior;
  if (R.ntiles == 0) return 0;
#define FA(NP) hipLaunchKernelGGL(k_fixrec_a<NP>, tile_grid(R), kTile, 0, s, L.k, F, flag, cluster, R)
  WITH_NP(L.k.np, FA)
#undef FA
  TICK("fix_recovery_a");
#define FB(NP) hipLaunchKernelGGL(k_fixrec_b<NP>, dim3(L.k.nplanes), dim3(64), 0, s, L.k, F, flag, cluster)
  WITH_NP(L.k.np, FB)
#undef FB
  TICK("fix_recovery_b");
  return PG_CHECK_LAUNCH();
}

int launch_exchange(const LaunchCtx &L, const KFields &F, double *const *flag, const int *nbr,
                    hipStream_t s) {
  if (L.ghosts.ntiles > 0) {
#define EX(NP) \
  hipLaunchKernelGGL(k_exchange<NP>, dim3(L.ghosts.ntiles), kTile, 0, s, L.k, F, flag, nbr, L.ghosts)
    WITH_NP(L.k.np, EX)
#undef EX
  }
  TICK("exchange");
  return PG_CHECK_LAUNCH();
}

int launch_bc(const LaunchCtx &L, const KFields &F, double *const *flag, hipStream_t s) {
  if (L.bcs.ntiles == 0) return 0;
#define BC(NP) hipLaunchKernelGGL(k_bc<NP>, dim3(L.bcs.ntiles), kTile, 0, s, L.k, F, flag, L.bcs)
  WITH_NP(L.k.np, BC)
#undef BC
  TICK("bc");
  return PG_CHECK_LAUNCH();
}

int launch_dt(const LaunchCtx &L, double *const *alfven, double *red, double *state,
              double dt_factor, double *est_out, hipStream_t s) {
  if (L.k.dtper == 1)
    hipLaunchKernelGGL(k_dt_reduce<1>, dim3(L.k.ndt), dim3(256), 0, s, L.k, alfven, red);
  else if (L.k.dtper == 4)
    hipLaunchKernelGGL(k_dt_reduce<4>, dim3(L.k.ndt), dim3(256), 0, s, L.k, alfven, red);
  else
    hipLaunchKernelGGL(k_dt_reduce<16>, dim3(L.k.ndt), dim3(256), 0, s, L.k, alfven, red);
  TICK("dt_reduce");
#define DF(W)                                                                                              \
  case W:                                                                                                 \
    hipLaunchKernelGGL(k_dt_final<W>, dim3(L.k.nmesh), dim3(1024), 0, s, L.k, red, state, dt_factor, est_out); \
    break;
  switch (L.dtlanes) { DF(1) DF(2) DF(4) DF(8) DF(16) DF(32) DF(64) }
#undef DF
  TICK("dt_final");
  return PG_CHECK_LAUNCH();
}

}  // namespace pangu
