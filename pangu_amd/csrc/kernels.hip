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

// ------------------------------------ flux divergence, update, source term
// dU/dt = -[sum_d (A_d F_d(+) - A_d F_d(-))]/V (Parthenon FluxDivergence),
// U(out) = U(init) + beta dt dU/dt (UpdateIndependentData) and the
// geometric source U_nu += beta dt sqrt|g| T^r_c Gamma^c_{nu r}
// (source_term.cc:171-228).  MODE: 1 = divergence only (writes dU/dt),
// 2 = update only (reads dU/dt), 3 = source only, 4 = all three fused.
// Flux divergence of one cell (and, for MODE 4, the update from the initial
// container) with the X2 / X3 terms present when D2 / D3.
// CTF: the face B fluxes are the constrained-transport values, formed here
// from edge EMFs that are themselves formed here from the Riemann B fluxes,
// exactly as k_emf and k_ct_faces would compute them (same operands, same
// operations), so neither CT kernel runs.  Each cell forms the 12 EMFs on
// its edges (each edge is shared by four cells; the extra arithmetic is
// cheaper than a kernel that writes and rereads the EMF arrays).  B
// components sit at packed indices 5..7.
template <bool D2, bool D3, int MODE, int NC, bool CTF>
__device__ __forceinline__ void flux_div(const DevBlock &B, const KFields &F0, const KFields &Finit,
                                         double *const *dudt, int b,
                                         int64_t id, int64_t sj, int64_t sk, double bdt,
                                         double unew[NC]) {
  const double a1 = B.dx[1] * B.dx[2], a2 = B.dx[0] * B.dx[2], a3 = B.dx[0] * B.dx[1];
  const double vol = B.dx[0] * B.dx[1] * B.dx[2];
  const double rvol = 1.0 / vol;
  double f1p[NC], f1m[NC], f2p[NC], f2m[NC], f3p[NC], f3m[NC], u0[NC];
  // Every access is base[u + id]: u is a workgroup-uniform offset (a row
  // sj, a plane sk, or 1) folded into the scalar base, id the cell.
  const uint32_t id32 = (uint32_t)id;
  auto at = [&](const double *p, int64_t u) { return ld32(p, u, id32); };
  // edge EMFs at uniform offset u from the cell, with the k_emf expressions
  const double *f1b2 = nullptr, *f1b3 = nullptr, *f2b1 = nullptr, *f2b3 = nullptr, *f3b1 = nullptr,
               *f3b2 = nullptr;
  if (CTF) {
    f1b2 = F0.flux[0][b * NC + 6];
    f1b3 = F0.flux[0][b * NC + 7];
    if (D2) {
      f2b1 = F0.flux[1][b * NC + 5];
      f2b3 = F0.flux[1][b * NC + 7];
    }
    if (D3) {
      f3b1 = F0.flux[2][b * NC + 5];
      f3b2 = F0.flux[2][b * NC + 6];
    }
  }
  auto E1 = [&](int64_t u) { return 0.25 * ((at(f2b3, u) + at(f2b3, u - sk)) - (at(f3b2, u) + at(f3b2, u - sj))); };
  auto E2 = [&](int64_t u) { return 0.25 * ((at(f3b1, u) + at(f3b1, u - 1)) - (at(f1b3, u) + at(f1b3, u - sk))); };
  auto E3 = [&](int64_t u) { return 0.25 * ((at(f1b2, u) + at(f1b2, u - sj)) - (at(f2b1, u) + at(f2b1, u - 1))); };
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int c = q - 5;  // B component when CTF and 0 <= c < 3
    const bool ctb = CTF && c >= 0 && c < 3;
    const double *f1 = F0.flux[0][b * NC + q];
    if (ctb && c == 0) {  // normal component: zero
      f1p[q] = 0;
      f1m[q] = 0;
    } else if (ctb && c == 1 && D2) {
      f1m[q] = 0.5 * (E3(0) + E3(sj));
      f1p[q] = 0.5 * (E3(1) + E3(1 + sj));
    } else if (ctb && c == 2 && D3) {
      f1m[q] = -0.5 * (E2(0) + E2(sk));
      f1p[q] = -0.5 * (E2(1) + E2(1 + sk));
    } else {
      f1p[q] = glb(f1)[id + 1];
      f1m[q] = glb(f1)[id];
    }
    if (D2) {
      const double *f2 = F0.flux[1][b * NC + q];
      if (ctb && c == 0) {
        f2m[q] = -0.5 * (E3(0) + E3(1));
        f2p[q] = -0.5 * (E3(sj) + E3(sj + 1));
      } else if (ctb && c == 1) {
        f2p[q] = 0.;
        f2m[q] = 0.;
      } else if (ctb && c == 2 && D3) {
        f2m[q] = 0.5 * (E1(0) + E1(sk));
        f2p[q] = 0.5 * (E1(sj) + E1(sj + sk));
      } else {
        f2p[q] = at(f2, sj);
        f2m[q] = at(f2, 0);
      }
    }
    if (D3) {
      const double *f3 = F0.flux[2][b * NC + q];
      if (ctb && c == 0) {
        f3m[q] = 0.5 * (E2(0) + E2(1));
        f3p[q] = 0.5 * (E2(sk) + E2(sk + 1));
      } else if (ctb && c == 1 && D2) {
        f3m[q] = -0.5 * (E1(0) + E1(sj));
        f3p[q] = -0.5 * (E1(sk) + E1(sk + sj));
      } else if (ctb && c == 2) {
        f3p[q] = 0;
        f3m[q] = 0;
      } else {
        f3p[q] = at(f3, sk);
        f3m[q] = at(f3, 0);
      }
    }
    if (MODE == 4) u0[q] = at(Finit.cons[b * NC + q], 0);
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    double s = (a1 * f1p[q] - a1 * f1m[q]);
    if (D2) s += (a2 * f2p[q] - a2 * f2m[q]);
    if (D3) s += (a3 * f3p[q] - a3 * f3m[q]);
    const double du = div_by(-s, vol, rvol);
    if (MODE == 1)
      glb(dudt[b * NC + q])[id] = du;
    else
      unew[q] = u0[q] + bdt * du;
  }
}

// Five waves per SIMD is the most the magnetised source-term variants reach
// without spilling (the field-free ones spill at five and run at four); the
// kernel is memory bound, so occupancy pays.
// One cell of k_div_update; the new U also goes to uout (when given).
// MF: form of the metric for the source term (FORM_FLAT: no source).
template <int MODE, int MF, bool HB, bool HK, bool CTF>
__device__ __forceinline__ void div_update_cell(const KCtx &C, const KFields &F0, const KFields &Finit,
                                                const KFields &F1, double *const *dudt,
                                                const double *dt_dev, double beta, double bdt_host,
                                                int b, int k, int j, int i, double *uout) {
  const DevBlock &B = C.blk[b];
  const int64_t sj = B.n[0], sk = (int64_t)B.n[0] * B.n[1];
  const int64_t id = k * sk + j * sj + i;
  constexpr int NC = ncomp<HB, HK>();
  const double bdt = dt_dev ? beta * dt_dev[2 * B.mesh] : bdt_host;
  double unew[NC];
  if (MODE == 1 || MODE == 4) {
    // one uniform branch on the block's active dimensions, so the loads of
    // all components sit in one basic block and overlap
    const bool d2 = B.n[1] > 1, d3 = B.n[2] > 1;
    if (d2 && d3)
      flux_div<true, true, MODE, NC, CTF>(B, F0, Finit, dudt, b, id, sj, sk, bdt, unew);
    else if (d2)
      flux_div<true, false, MODE, NC, CTF>(B, F0, Finit, dudt, b, id, sj, sk, bdt, unew);
    else if (d3)
      flux_div<false, true, MODE, NC, CTF>(B, F0, Finit, dudt, b, id, sj, sk, bdt, unew);
    else
      flux_div<false, false, MODE, NC, CTF>(B, F0, Finit, dudt, b, id, sj, sk, bdt, unew);
  } else if (MODE == 2) {
#pragma unroll
    for (int q = 0; q < NC; ++q)
      unew[q] = glb(Finit.cons[b * NC + q])[id] + bdt * glb(dudt[b * NC + q])[id];
  } else {
#pragma unroll
    for (int q = 0; q < NC; ++q) unew[q] = glb(F1.cons[b * NC + q])[id];
  }
  if (MODE == 1) return;
  if (MF != FORM_FLAT && (MODE == 3 || MODE == 4)) {
    const DevGeo &G = C.geo[B.geo];
    const int64_t t = cen_index(G, k, j, i);
    CenLoad m;
    load_cen_state<MF>(G, t, m);
    double p[NPRIM];
#pragma unroll
    for (int s = 0; s < NPRIM; ++s) p[s] = 0.0;
#pragma unroll
    for (int q = 0; q < NC; ++q) p[slot_of<HB, HK>(q)] = glb(F1.prim[b * NC + q])[id];
    St s;
    calc_state<MF, HB>(p, m.g, m.gc0, m.alpha, s);
    const double gam = C.ph.gamma;
    const double pg = (gam - 1.) * p[ENY];
    const double h = p[RHO] + gam * p[ENY];
    const double etot = HB ? h + s.bsq : h, ptot = HB ? pg + 0.5 * s.bsq : pg;
    double T[4][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      T[0][c] = tmunu<0, HB>(s, etot, ptot, c);
      T[1][c] = tmunu<1, HB>(s, etot, ptot, c);
      T[2][c] = tmunu<2, HB>(s, etot, ptot, c);
      T[3][c] = tmunu<3, HB>(s, etot, ptot, c);
    }
    // one scalar base for the connection block (40 or 64 slots) and a
    // 32-bit index per slot: per-slot scalar bases would exhaust the scalar
    // registers
    const double *conn = G.cen + (int64_t)CG_CONN * G.ncen;
    const uint32_t ncen32 = (uint32_t)G.ncen, t32 = (uint32_t)t;
    const bool sym = G.conn_sym != 0;
#pragma unroll
    for (int dd = 0; dd < 4; ++dd) {
      double con = 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int slot = sym ? 10 * c + conn_pair(dd, r) : 16 * c + 4 * dd + r;
          con += T[r][c] * ldc32(conn, 0, (uint32_t)slot * ncen32 + t32);
        }
      const int q = (dd == 0) ? 1 : 1 + dd;
      unew[q] += con * m.sg * bdt;
    }
  }
  if (uout) {
    // the caller goes on with the values; memory is next read a stage later
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      stnt32(F1.cons[b * NC + q], (uint32_t)id, unew[q]);
      uout[q] = unew[q];
    }
  } else {
    // the next kernel (the source term, the recovery) reads them: with stores
    // past L2 the tasks from flux divergence to source took 53.1 us for 64^3
    // cells in MKS instead of 50.1
#pragma unroll
    for (int q = 0; q < NC; ++q) glb(F1.cons[b * NC + q])[id] = unew[q];
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

// -------------------------------------------------- recovery (+ heating)
// ApplyElectronHeating (electron_heating.cc:66-109) on one recovered cell
// from its primitives p (rho, u, u~, B and the stale entropy; K_e is not
// read); the centre metric is loaded here.
template <int MF, bool HB, bool HK>
__device__ __forceinline__ void heat_vals(const KCtx &C, const KFields &F, const DevGeo &G, int64_t t,
                                          int b, int64_t id, const Arr32<double> *pp,
                                          const double p[NPRIM], const double *ureg = nullptr) {
  constexpr int NC = ncomp<HB, HK>();
  CenLoad m;
  load_cen_state<MF>(G, t, m);
  St s;
  calc_state<MF, HB>(p, m.g, m.gc0, m.alpha, s);
  const uint32_t id32 = (uint32_t)id;
  // conserved components: from memory, or from registers (ureg, in
  // component order) when the caller has just written them
  auto cu = [&](int q) { return ureg ? ureg[q] : ld32(F.cons[b * NC + q], 0, id32); };
  const double crho = cu(0);
  HeatIn c;
  c.rho = p[RHO];
  c.energy = p[ENY];
  c.bsq = s.bsq;
  c.adv_total = cu(ient<HB>()) / crho;
  c.rec_total = p[ENT];
  c.adv_e = cu(ikel<HB>()) / crho;
  pp[ikel<HB>()][id] = heat_apply(C.ph, c);
}

// The same with the primitives read from memory.
template <int MF, bool HB, bool HK>
__device__ __forceinline__ void heat_cell(const KCtx &C, const KFields &F, const DevGeo &G, int64_t t,
                                          int b, int64_t id, const Arr32<double> *pp) {
  constexpr int NC = ncomp<HB, HK>();
  double p[NPRIM];
#pragma unroll
  for (int s = 0; s < NPRIM; ++s) p[s] = 0.0;
#pragma unroll
  for (int q = 0; q < NC; ++q) p[slot_of<HB, HK>(q)] = pp[q][id];
  heat_vals<MF, HB, HK>(C, F, G, t, b, id, pp, p);
}

// The centre metric the recovery reads, as far as form MF leaves it open
// (gcon is not symmetric bit for bit, so each open entry is read), sqrt|g|
// and 1/sqrt(-g^00).
template <int MF>
__device__ __forceinline__ void load_cen_metric(const DevGeo &G, int64_t t, CenMetric &m, double &sg,
                                                double &alpha) {
  auto comp = [&](int n) { return ldc32(G.cen, (int64_t)n * G.ncen, (uint32_t)t); };
  double gc0[4];
  load_metric<MF, CG_GCON, CG_ALPHA>(comp, m.gcov, gc0, alpha);
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      m.gcon[4 * r + c] = MF == FORM_FLAT ? m.gcov[4 * r + c] : g_open<MF>(r, c) ? comp(CG_GCON + 4 * r + c) : 0.0;
  m.lapse = MF == FORM_FLAT ? 1.0 : comp(CG_LAPSE);
  sg = MF == FORM_FLAT ? 1.0 : comp(CG_SG);
}

// Recovery (invertor.cc:184-319) and, when HEAT, ApplyElectronHeating
// (electron_heating.cc:66-109) on the recovered cell.  REC: 0 chainer,
// 1 Kastaun, 2 1Dvsq alone, -1 none (heating only).
template <int MF, int REC, bool HB, bool HK, bool HEAT>
__device__ __forceinline__ void recover_cell(const KCtx &C, const KFields &F, const SharedTabs &S, int b,
                                             int k, int j, int i, double x0 = -1.0,
                                             const double *ureg = nullptr) {
  const DevBlock &B = C.blk[b];
  const int64_t id = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  constexpr int NC = ncomp<HB, HK>();
  const DevGeo &G = C.geo[B.geo];
  const int64_t t = cen_index(G, k, j, i);
  const Phys &P = C.ph;
  Arr32<double> pp[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) pp[q] = Arr32<double>{F.prim[b * NC + q]};
  if (REC >= 0) {
    const bool chainer = (REC != 1);
    bool excised = false;
    if (P.metric == PANGU_METRIC_CKS && ldc32(G.cen, (int64_t)CG_RAD * G.ncen, (uint32_t)t) < P.r_excise) excised = true;
    if (excised) {
      if (chainer && S.flag) glb(S.flag[b])[id] = 0.0;
      if (S.status) glb(S.status[b])[id] = -1;
      if (S.iters) glb(S.iters[b])[id] = 0;
    } else {
      CenMetric m;
      double sg, alpha;
      load_cen_metric<MF>(G, t, m, sg, alpha);
      double U[9], Ph[9], bnew[3] = {0.0, 0.0, 0.0};
      Arr32<double> cons[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) cons[q] = Arr32<double>{F.cons[b * NC + q]};
      // U from memory, or from registers (ureg) when the update just wrote it
      auto cv = [&](int q) { return ureg ? ureg[q] : (double)cons[q][id]; };
      const double c_rho = cv(0), c_eny = cv(1);
      const double isg = 1.0 / sg;
      const double aos = alpha * isg;
      U[RHO] = aos * c_rho;
      U[ENY] = aos * (c_eny - c_rho);
      U[UX1] = aos * cv(2);
      U[UX2] = aos * cv(3);
      U[UX3] = aos * cv(4);
      if (HB) {
        const double cb1 = cv(5), cb2 = cv(6), cb3 = cv(7);
        U[BX1] = aos * cb1;
        U[BX2] = aos * cb2;
        U[BX3] = aos * cb3;
        bnew[0] = cb1 * isg;
        bnew[1] = cb2 * isg;
        bnew[2] = cb3 * isg;
        pp[5][id] = bnew[0];
        pp[6][id] = bnew[1];
        pp[7][id] = bnew[2];
      } else {
        U[BX1] = 0.0;
        U[BX2] = 0.0;
        U[BX3] = 0.0;
      }
      U[ENT] = aos * cv(ient<HB>());
      // the Newton schemes start from the previous primitives; Kastaun's
      // bracket needs none (it writes rho, u and u~ only on success), so
      // their loads are skipped
#pragma unroll
      for (int s = 0; s < 9; ++s) Ph[s] = 0.0;
      if (REC != 1) {
        Ph[RHO] = pp[0][id];
        Ph[ENY] = pp[1][id];
        Ph[UX1] = pp[2][id];
        Ph[UX2] = pp[3][id];
        Ph[UX3] = pp[4][id];
        Ph[ENT] = pp[ient<HB>()][id];
      }
      int st = 0, it = 0, itn = 0;
      bool write = true;
      if (REC == 1) {
        double mu = 0.0;
        st = c2p_kastaun<MF>(U, Ph, P.gamma, m, it, &mu);
        if (S.root) glb(S.root[b])[id] = (st == 0) ? mu : __builtin_nan("");
        itn = it;
        write = (st == 0);
      } else if (REC == 2) {
        // x0 >= 0: the learned start (k_recover_learned_vsq)
        st = c2p_1dvsq<MF>(U, Ph, P.gamma, m, it, x0);
        itn = it;
      } else {
        st = c2p_2d<MF>(U, Ph, P.gamma, m, it);
        itn = it;
        if (st != 0) {
          st = c2p_1dvsq<MF>(U, Ph, P.gamma, m, it);
          itn += it;
          if (st != 0) {
            st = c2p_1d<MF>(U, Ph, P.gamma, m, it);
            itn += it;
          }
        }
      }
      if (chainer && S.flag) {
        const double fv = (st == 0) ? 1.0 : 0.0;
        glb(S.flag[b])[id] = fv;
        if (S.flag_rec) glb(S.flag_rec[b])[id] = fv;
      }
      if (S.status) glb(S.status[b])[id] = st;
      if (S.iters) glb(S.iters[b])[id] = itn;
      if (write) {
        pp[0][id] = Ph[RHO];
        pp[1][id] = Ph[ENY];
        pp[2][id] = Ph[UX1];
        pp[3][id] = Ph[UX2];
        pp[4][id] = Ph[UX3];
      }
      if (HEAT && HK) {
        // the heating reads the primitives just written from registers (the
        // compiler cannot forward them: the stores may alias other arrays);
        // a cell whose recovery failed keeps its previous primitives
        double hp[NPRIM];
#pragma unroll
        for (int s = 0; s < NPRIM; ++s) hp[s] = 0.0;
        if (write) {
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
          hp[BX1] = bnew[0];
          hp[BX2] = bnew[1];
          hp[BX3] = bnew[2];
        }
        hp[ENT] = pp[ient<HB>()][id];
        heat_vals<MF, HB, HK>(C, F, G, t, b, id, pp, hp, ureg);
        return;
      }
    }
  }
  if (HEAT && HK) heat_cell<MF, HB, HK>(C, F, G, t, b, id, pp);
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
#define RQ(MF_, R_, HB_, HK_, HE_)                                                                    \
  hipLaunchKernelGGL((k_recover_queue<MF_, R_, HB_, HK_, HE_>),                                       \
                     dim3(resident_groups(k_recover_queue<MF_, R_, HB_, HK_, HE_>, R.tile, R.ntiles)), \
                     wg, 0, s, L.k, F, S, R, L.queue)
#define RC(R_, HB_, HK_, HE_)                                                                        \
  if ((R_ == 1 && W && W->kind == 0) || (R_ == 2 && W && W->kind == 1)) {                             \
    if (mf == FORM_NULLV)                                                                             \
      launch_learned<FORM_NULLV, HB_, HK_, HE_>(L, F, S, *W, R, g, wg, s, upd);                       \
    else                                                                                              \
      launch_learned<FORM_FULL, HB_, HK_, HE_>(L, F, S, *W, R, g, wg, s, upd);                        \
  } else if (persist && mf == FORM_NULLV)                                                             \
    RQ(FORM_NULLV, R_, HB_, HK_, HE_);                                                                \
  else if (persist)                                                                                   \
    RQ(FORM_FULL, R_, HB_, HK_, HE_);                                                                 \
  else if (mf == FORM_POLOIDAL)                                                                       \
    hipLaunchKernelGGL((k_recover<FORM_POLOIDAL, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R);     \
  else if (mf == FORM_FLAT)                                                                           \
    hipLaunchKernelGGL((k_recover<FORM_FLAT, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R);         \
  else                                                                                                \
    hipLaunchKernelGGL((k_recover<FORM_NULLV, R_, HB_, HK_, HE_>), g, wg, 0, s, L.k, F, S, R)
#define RC2(R_, HE_)                          \
  if (hb && hk) { RC(R_, true, true, HE_); }  \
  else if (hb) { RC(R_, true, false, HE_); }  \
  else if (hk) { RC(R_, false, true, HE_); }  \
  else { RC(R_, false, false, HE_); }
  const bool h = heat && hk;
  if (rec == 0) {
    if (h) { RC2(0, true) } else { RC2(0, false) }
  } else if (rec == 1) {
    if (h) { RC2(1, true) } else { RC2(1, false) }
  } else if (rec == 2) {
    if (h) { RC2(2, true) } else { RC2(2, false) }
  } else if (h) {
    RC2(-1, true)
  }
#undef RC2
#undef RC
#undef RQ
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
