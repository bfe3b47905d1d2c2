// Device code of the same-level ghost exchange and of cell copies.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "kernels.h"

namespace pangu {

// Ghost cell g of a block, numbered over three slabs: the k-ghost planes
// (full j, i extent), then the j-ghost rows of interior planes (full i),
// then the i-ghost cells of interior rows.  Every ghost cell appears once,
// with i fastest inside each slab.
__device__ __forceinline__ void ghost_cell(const DevBlock &B, int g, int &k, int &j, int &i) {
  const int n0 = B.n[0], n1 = B.n[1], n2 = B.n[2];
  const int a2 = B.s[2] + (n2 - 1 - B.e[2]);
  const int A = a2 * n1 * n0;
  if (g < A) {
    const int kk = g / (n1 * n0), r = g - kk * n1 * n0;
    k = kk < B.s[2] ? kk : B.e[2] + 1 + (kk - B.s[2]);
    j = r / n0;
    i = r - j * n0;
    return;
  }
  g -= A;
  const int b1 = B.s[1] + (n1 - 1 - B.e[1]);
  const int nk = B.e[2] - B.s[2] + 1;
  const int Bc = nk * b1 * n0;
  if (g < Bc) {
    const int kk = g / (b1 * n0), r = g - kk * b1 * n0;
    const int jj = r / n0;
    k = B.s[2] + kk;
    j = jj < B.s[1] ? jj : B.e[1] + 1 + (jj - B.s[1]);
    i = r - jj * n0;
    return;
  }
  g -= Bc;
  const int nj = B.e[1] - B.s[1] + 1;
  const int c0 = B.s[0] + (n0 - 1 - B.e[0]);
  const int kk = g / (nj * c0), r = g - kk * nj * c0;
  const int jj = r / c0, ii = r - jj * c0;
  k = B.s[2] + kk;
  j = B.s[1] + jj;
  i = ii < B.s[0] ? ii : B.e[0] + 1 + (ii - B.s[0]);
}

// Copies the NP packed components (and the flag) of cell src of block sb to
// cell dst of block db, with the sign of the components in flip (bit q)
// changed.  Every pointer and value is loaded before the first store: a
// store may alias the pointer tables and the other arrays, so a loop of
// load / store pairs waits for memory twice per component.  With the three
// boundary passes in one launch (k_bc): cycle of eight 32x16x16 torus blocks
// about 195 -> 170 us, 2-D torus 512x256 227 -> 210 us, Orszag-Tang 256^2
// 109 -> 104 us, refined mesh (k_xfill, k_xprol) 424 -> 388 us.
template <int NP>
__device__ __forceinline__ void copy_cell(const KFields &F, double *const *flag, int db, int64_t dst, int sb,
                                          int64_t src, unsigned flip) {
  double *to[NP];
  double v[NP], fl = 0.0;
#pragma unroll
  for (int q = 0; q < NP; ++q) to[q] = F.prim[db * NP + q];
#pragma unroll
  for (int q = 0; q < NP; ++q) v[q] = glb(F.prim[sb * NP + q])[src];
  double *const tf = flag ? flag[db] : nullptr;
  if (flag) fl = glb(flag[sb])[src];
#pragma unroll
  for (int q = 0; q < NP; ++q) glb(to[q])[dst] = ((flip >> q) & 1) ? -v[q] : v[q];
  if (flag) glb(tf)[dst] = fl;
}

// Same-level exchange: a ghost cell of block b takes the interior value of
// the neighbour in its offset direction (periodic wrap encoded in nbr).
// g: ghost cell of block b.
template <int NP>
__device__ __forceinline__ void exchange_cell(const KCtx &C, const KFields &F, double *const *flag,
                                              const int *nbr, int b, int g) {
  const DevBlock &B = C.blk[b];
  const int interior = (B.e[0] - B.s[0] + 1) * (B.e[1] - B.s[1] + 1) * (B.e[2] - B.s[2] + 1);
  if (g >= (int)B.ncell - interior) return;
  int k, j, i;
  ghost_cell(B, g, k, j, i);
  const int o0 = (i < B.s[0]) ? -1 : (i > B.e[0] ? 1 : 0);
  const int o1 = (j < B.s[1]) ? -1 : (j > B.e[1] ? 1 : 0);
  const int o2 = (k < B.s[2]) ? -1 : (k > B.e[2] ? 1 : 0);
  if ((o0 | o1 | o2) == 0) return;
  const int nb = nbr[b * 27 + (o2 + 1) * 9 + (o1 + 1) * 3 + (o0 + 1)];
  if (nb < 0) return;
  // blocks of one mesh share one shape, so the neighbour's strides are B's
  const int si = i - o0 * (B.e[0] - B.s[0] + 1);
  const int sj = j - o1 * (B.e[1] - B.s[1] + 1);
  const int sk = k - o2 * (B.e[2] - B.s[2] + 1);
  const int64_t dst = ((int64_t)k * B.n[1] + j) * B.n[0] + i;
  const int64_t src = ((int64_t)sk * B.n[1] + sj) * B.n[0] + si;
  copy_cell<NP>(F, flag, b, dst, nb, src, 0u);
}

}  // namespace pangu
