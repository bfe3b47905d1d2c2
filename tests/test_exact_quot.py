"""quot and root of exact_div.h on the CPU: the steps after the hardware's
first approximation return the IEEE quotient and square root for any seed as
good as the hardware's (relative error up to 2^-23 here), over the exponent
range the header states, and a seed or step that is too poor is noticed."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pangu_amd", "csrc")

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
static double noise();
#define PANGU_SEED_RCP(y) ((1.0 / (y)) * (1.0 + noise()))
#define PANGU_SEED_RSQ(x) ((1.0 / std::sqrt(x)) * (1.0 + noise()))
#include "exact_div.h"
static uint64_t st = 88172645463325252ull;
static uint64_t rnd() { st ^= st << 13; st ^= st >> 7; st ^= st << 17; return st; }
static double unit() { return (rnd() >> 11) * 0x1p-53; }
static double noise() { return (2.0 * unit() - 1.0) * SEED_ERROR; }
static double draw(int e) {
  // significands dense, sparse and next to 1 and 2, exponents within +-e
  uint64_t m = rnd() >> 12;
  switch (rnd() % 4) {
    case 0: m &= ~0ull << (rnd() % 52); break;
    case 1: m >>= rnd() % 52; break;
    case 2: m = 0xfffffffffffffull - (m >> (rnd() % 52)); break;
  }
  // an all-ones significand is excepted (exact_div.h): clear its last bit
  if (m == 0xfffffffffffffull) m ^= 1;
  double s;
  const uint64_t b = (1023ull << 52) | m;
  std::memcpy(&s, &b, 8);
  return std::ldexp(s, (int)(rnd() % (2 * e + 1)) - e);
}
int main() {
  long bad = 0;
  for (long n = 0; n < 6000000; ++n) {
    const double x = (rnd() & 1 ? -1.0 : 1.0) * draw(440), y = (rnd() & 1 ? -1.0 : 1.0) * draw(440);
    if (pangu::quot(x, y) != x / y) ++bad;
    const double z = draw(740);
    if (pangu::root(z) != std::sqrt(z)) ++bad;
    // squares and their neighbours: results next to a tie or exact
    const double w = draw(300), q = std::nextafter(w * w, (rnd() & 1) ? 0.0 : 1e300);
    if (pangu::root(w * w) != std::sqrt(w * w) || pangu::root(q) != std::sqrt(q)) ++bad;
    if (pangu::quot(w * y, y) != (w * y) / y) ++bad;
  }
  // the excepted divisor: within one unit in the last place
  for (long n = 0; n < 100000; ++n) {
    const double x = draw(300), y = std::nextafter(2.0, 0.0), q = x / y, d = pangu::quot(x, y);
    if (d != q && d != std::nextafter(q, 0.0) && d != std::nextafter(q, 1e308)) ++bad;
  }
  if (pangu::quot(0.0, 3.0) != 0.0 || !std::isnan(pangu::root(-1.0))) ++bad;
  std::printf("%ld\n", bad);
  return 0;
}
"""


def _bad(tmp_path, seed_error, edit=None):
    hdr = open(os.path.join(CSRC, "exact_div.h")).read()
    if edit:
        assert edit[0] in hdr
        hdr = hdr.replace(edit[0], edit[1])
    (tmp_path / "exact_div.h").write_text(hdr)
    (tmp_path / "q.cpp").write_text(SRC)
    exe = str(tmp_path / "q")
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    subprocess.run([gxx, "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", f"-DSEED_ERROR={seed_error}",
                    "-I", str(tmp_path), str(tmp_path / "q.cpp"), "-o", exe], check=True)
    return int(subprocess.run([exe], check=True, capture_output=True, text=True).stdout)


@pytest.mark.parametrize("seed_error", ["0x1p-23", "0x1p-28"])
def test_quot_and_root_are_ieee(tmp_path, seed_error):
    assert _bad(tmp_path, seed_error) == 0


def test_missing_newton_step_is_caught(tmp_path):
    step = "  r = fma(r, fma(-y, r, 1.0), r);\n"
    assert _bad(tmp_path, "0x1p-23", (step + step, step)) > 0


def test_missing_root_steps_are_caught(tmp_path):
    steps = "  s = fma(s, e, s);\n  s = fma(fma(-s, s, x), h, s);\n"
    assert _bad(tmp_path, "0x1p-23", (steps, "")) > 0
