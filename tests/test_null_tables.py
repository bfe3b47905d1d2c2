"""The xi and l tables of Cartesian Kerr-Schild (fill_null_table) on the CPU:
gcov = eta + (xi l_r) l_c, formed as the kernels form it (gcov_from_null),
equals the centre and face tables' gcov bit for bit, entry by entry, for
blocks of one to three dimensions."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pangu_amd", "csrc")

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "common.h"
#include "host.h"
using namespace pangu;
int main(int argc, char **argv) {
  pangu_config cfg;
  std::memset(&cfg, 0, sizeof(cfg));
  cfg.metric = PANGU_METRIC_CKS;
  cfg.a = std::atof(argv[1]);
  cfg.h = 0.3;
  pangu_block B;
  std::memset(&B, 0, sizeof(B));
  const double lo[3] = {2.3, -1.7, 0.25}, w[3] = {1.1, 2.9, 0.5};
  for (int d = 0; d < 3; ++d) {
    B.nx[d] = std::atoi(argv[2 + d]);
    B.ng[d] = B.nx[d] > 1 ? 4 : 0;
    B.xmin[d] = lo[d];
    B.dx[d] = w[d] / B.nx[d];
  }
  const HostBlock H = make_host_block(B);
  const bool has3d = H.n[2] > 1;
  const int shift = std::atoi(argv[5]);  // entries the null table is read off by
  long bad = 0, all = 0;
  for (int d = 0; d < 4; ++d) {  // 3: centres
    if (d < 3 && (H.n[d] == 1 || (d == 2 && !has3d))) continue;
    const int fi = H.n[0] + (d == 0), fj = H.n[1] + (d == 1), fk = has3d ? H.n[2] + (d == 2) : 1;
    const int64_t n = (int64_t)fi * fj * fk;
    std::vector<double> tab((size_t)(n * (d == 3 ? (int)CG_NCOMP : (int)FG_NCOMP))), nul((size_t)(4 * n + 4));
    if (d == 3)
      geom::fill_centre_table(cfg, H, fi, fj, fk, has3d, tab.data());
    else
      geom::fill_face_table(cfg, H, d, fi, fj, fk, has3d, tab.data());
    geom::fill_null_table(cfg, H, d, fi, fj, fk, has3d, nul.data());
    for (int64_t e = 0; e < n; ++e) {
      double l[4] = {1.0, 0.0, 0.0, 0.0};
      const double xi = nul[(size_t)(e + shift)];
      for (int q = 1; q < 4; ++q) l[q] = nul[(size_t)(q * n + e + shift)];
      for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
          const double t = r ? xi * l[r] : xi, u = c ? t * l[c] : t;
          const double g = r != c ? u : (r ? 1.0 : -1.0) + u;
          const double want = tab[(size_t)((4 * r + c) * n + e)];
          ++all;
          if (std::memcmp(&g, &want, sizeof(g)) != 0) ++bad;
        }
    }
  }
  std::printf("%ld %ld\n", bad, all);
  return 0;
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("null_tables")
    (d / "n.cpp").write_text(SRC)
    out = str(d / "n")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fopenmp", "-ffp-contract=off", f"-I{CSRC}", str(d / "n.cpp"),
                    os.path.join(CSRC, "geometry.cpp"), os.path.join(CSRC, "problems.cpp"), "-o", out],
                   check=True, capture_output=True)
    return out


def _run(exe, a, nx, shift=0):
    r = subprocess.run([exe, str(a), *map(str, nx), str(shift)], check=True, capture_output=True, text=True)
    return tuple(int(x) for x in r.stdout.split())


@pytest.mark.parametrize("a", [0.9375, 0.0, -0.5])
@pytest.mark.parametrize("nx", [(12, 9, 7), (31, 20, 1), (50, 1, 1)])
def test_gcov_from_null_equals_the_tables(exe, a, nx):
    bad, n = _run(exe, a, nx)
    assert n > 0 and bad == 0


def test_a_misplaced_entry_is_caught(exe):
    bad, n = _run(exe, 0.9375, (12, 9, 7), shift=1)
    assert bad > n // 2
