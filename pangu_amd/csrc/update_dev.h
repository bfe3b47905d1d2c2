// Device code of one cell's update (flux divergence, RK update, geometric
// source) and of its recovery and electron heating.
#pragma once
#include <hip/hip_runtime.h>
#include <float.h>

#include "cell_dev.h"
#include "common.h"
#include "kernels.h"
#include "physics_dev.h"
#include "recovery_dev.h"

namespace pangu {

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

}  // namespace pangu
