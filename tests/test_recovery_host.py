"""The recovery schemes of recovery_dev.h, compiled for the host, against the
oracle's on the CPU: status, step count and primitives bit for bit, in the
forms the kernels are compiled for, over consistent, perturbed and hopeless
states from 1e-100 to 1e100, flat and Cartesian Kerr-Schild.  (The seeds of
quot and root are exact here; tests/test_exact_quot.py covers the rest.)"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_py as O
from pangu_amd import abi, configs
from test_exact_div import CLANG
from test_recovery_vsq1_gpu import GAMMA, STATES, _state

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pangu_amd", "csrc")

STUB = r"""
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
using std::isfinite;
#define __device__
#define __host__
#define __forceinline__ inline
"""
SRC = r"""
#include <cstring>
#include "recovery_dev.h"
using namespace pangu;
template <int MF>
static int solve(int scheme, const double *U, double *p, double gamma, const CenMetric &m, int *it) {
  return scheme == 0   ? c2p_2d<MF>(U, p, gamma, m, *it)
         : scheme == 1 ? c2p_1dvsq<MF>(U, p, gamma, m, *it)
         : scheme == 2 ? c2p_1d<MF>(U, p, gamma, m, *it)
                       : c2p_kastaun<MF>(U, p, gamma, m, *it);
}
extern "C" int c2p(int form, int scheme, const double *U, double *p, double gamma, const double *gcov,
                   const double *gcon, int *it) {
  CenMetric m;
  std::memcpy(m.gcov, gcov, sizeof(m.gcov));
  std::memcpy(m.gcon, gcon, sizeof(m.gcon));
  m.lapse = std::sqrt(-1.0 / gcon[0]);
  return form == FORM_FLAT    ? solve<FORM_FLAT>(scheme, U, p, gamma, m, it)
         : form == FORM_NULLV ? solve<FORM_NULLV>(scheme, U, p, gamma, m, it)
                              : solve<FORM_FULL>(scheme, U, p, gamma, m, it);
}
"""
FULL, FLAT, NULLV = 0, 2, 3
ETA = np.diag([-1.0, 1.0, 1.0, 1.0])


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("ROCm clang++ not present")
    d = tmp_path_factory.mktemp("recovery_host")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    (d / "r.cpp").write_text(SRC)
    out = str(d / "r.so")
    subprocess.run([CLANG, "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-fPIC", "-shared", "-D__HIPCC__",
                    f"-I{d}", f"-I{CSRC}", str(d / "r.cpp"), "-o", out], check=True, capture_output=True)
    return C.CDLL(out)


def _solve(lib, form, scheme, U, p, gcov, gcon):
    dp = C.POINTER(C.c_double)
    q, it = p.copy(), C.c_int()
    a = [np.ascontiguousarray(x, dtype=np.float64) for x in (U, gcov, gcon)]
    st = lib.c2p(form, scheme, a[0].ctypes.data_as(dp), q.ctypes.data_as(dp), C.c_double(GAMMA),
                 a[1].ctypes.data_as(dp), a[2].ctypes.data_as(dp), C.byref(it))
    return st, q, it.value


def _states(n, scale, seed, gcov, gcon):
    rng = np.random.default_rng(seed)
    alpha = np.sqrt(-1.0 / gcon[0, 0])
    for _ in range(n):
        s = 10.0 ** rng.uniform(-scale, scale)
        p = np.zeros(10)
        p[0] = s * 10 ** rng.uniform(-3, 3)
        p[1] = p[0] * 10 ** rng.uniform(-6, 4)
        p[2:5] = rng.normal(size=3) * 10 ** rng.uniform(-3, 1)
        if rng.random() < 0.7:
            p[5:8] = rng.normal(size=3) * np.sqrt(p[0]) * 10 ** rng.uniform(-3, 2)
        p[8] = (GAMMA - 1.0) * p[1] * p[0] ** -GAMMA
        U = alpha * O.flux(GAMMA, p, gcov, gcon, -1.0, 0)[:9]  # up to sqrt|g| = 1 here
        U[1] -= U[0]
        kind = rng.random()
        if kind > 0.4:
            U[1:5] *= 1.0 + rng.normal(size=4) * 10 ** rng.uniform(-6, 0)
        g = p[:9].copy()
        g[1] *= 10 ** rng.uniform(-1, 1)
        g[2:5] *= rng.uniform(0.8, 1.2)
        if kind > 0.7:
            g[8] *= 10 ** rng.uniform(-6, 6)
        yield U, g


def _cks_point():
    """gcov and gcon at a point where no two mirrored entries of gcov agree."""
    d = configs.orszag_tang(16, (1, 1, 1))
    d.update(metric=configs.METRIC["cks"], a=0.9375)
    cfg, dp = abi.config_from(d), C.POINTER(C.c_double)
    rng = np.random.default_rng(1)
    while True:
        x = np.concatenate([[0.0], rng.uniform(-4.0, 4.0, 3)])
        c = np.zeros(abi.CENTRE_NCOMP)
        assert abi.lib().pangu_geometry_entry(C.byref(cfg), 0, x.ctypes.data_as(dp), c.ctypes.data_as(dp)) == abi.OK
        g = c[:16].reshape(4, 4)
        if g[1, 2] != g[2, 1] and g[1, 3] != g[3, 1] and g[2, 3] != g[3, 2] and np.linalg.norm(x) > 3.0:
            return g.copy(), c[16:32].reshape(4, 4).copy()


@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
@pytest.mark.parametrize("metric", ["flat", "cks"])
def test_schemes_equal_the_oracle_bit_for_bit(lib, scheme, metric):
    gcov, gcon = (ETA, ETA) if metric == "flat" else _cks_point()
    solved = 0
    for scale in (0.0, 8.0, 100.0):
        for U, g in _states(1500, scale, 17 + scheme, gcov, gcon):
            want = O.c2p(scheme, U, g, GAMMA, gcov, gcon)
            solved += want[0] == 0
            for form in (FULL, FLAT if metric == "flat" else NULLV):
                got = _solve(lib, form, scheme, U, g, gcov, gcon)
                assert (got[0], got[2]) == (want[0], want[2]), (U, g)
                if want[0] == 0:  # (the entropy is formed by the caller)
                    assert np.array_equal(got[1][:5], want[1][:5]), (U, g)
    assert 500 < solved < 4500


def test_an_iterate_at_the_speed_of_light(lib):
    for words in STATES:
        u, p = _state(words)
        U = np.append(u, p[8] * u[0])
        assert _solve(lib, FLAT, 0, U, p, ETA, ETA)[0] == 4
