"""Structure of the geometry tables that the kernels of each metric form rely
on (physics_dev.h, MetricForm): which entries are exactly zero, one or equal
to their transpose, checked bit for bit over each metric's domain and on the
polar axis."""
import ctypes as C

import numpy as np
import pytest

from pangu_amd import abi, configs


def _tables(kind, n=400):
    L = abi.lib()
    d = configs.torus2d(64, 32)
    d["metric"] = abi.METRIC[kind]
    rng = np.random.default_rng(7)
    dp = C.POINTER(C.c_double)
    cen, face, xs, spins = [], [], [], []
    for a, h in ((0.9375, 0.3), (0.0, 0.0), (-0.5, 0.9)):
        d.update(a=a, h=h)
        cfg = abi.config_from(d)
        for m in range(n):
            if kind == "cks":
                x = np.concatenate([[0.0], rng.uniform(-30.0, 30.0, 3)])
            else:
                x = np.array([0.0, rng.uniform(-0.6, 4.0), rng.uniform(-1.1, 1.1), rng.uniform(0.0, 6.3)])
                if m < 4:
                    x[2] = (-1.0, 1.0, 0.0, -1.0 + 1e-9)[m]
            c = np.zeros(abi.CENTRE_NCOMP)
            assert L.pangu_geometry_entry(C.byref(cfg), 0, x.ctypes.data_as(dp), c.ctypes.data_as(dp)) == abi.OK
            cen.append(c)
            xs.append(x)
            spins.append(a)
            for dd in (1, 2, 3):
                f = np.zeros(abi.FACE_NCOMP)
                assert L.pangu_geometry_entry(C.byref(cfg), dd, x.ctypes.data_as(dp), f.ctypes.data_as(dp)) == abi.OK
                face.append(f)
    return np.array(cen), np.array(face), xs, spins


def _points(kind):
    cen, _, xs, spins = _tables(kind)
    return xs, spins, cen


@pytest.mark.parametrize("kind", ["mks", "bl", "cks", "minkowski"])
def test_tables_have_the_metric_form(kind):
    cen, face, _, _ = _tables(kind)
    for tab, g00 in ((cen, cen[:, 16:20]), (face, face[:, 16:20])):
        g = tab[:, :16].reshape(-1, 4, 4)
        # every form: the time row equals the time column
        assert np.array_equal(g[:, 0, :], g[:, :, 0])
        if kind == "cks":
            continue
        assert np.array_equal(g, g.transpose(0, 2, 1))
        for m in (0, 1, 3):
            assert np.all(g[:, m, 2] == 0.0) and np.all(g[:, 2, m] == 0.0)
        assert np.all(g00[:, 2] == 0.0)
        if kind == "minkowski":
            assert np.array_equal(g, np.broadcast_to(np.diag([-1.0, 1.0, 1.0, 1.0]), g.shape))
            assert np.array_equal(g00, np.broadcast_to([-1.0, 0.0, 0.0, 0.0], g00.shape))
    if kind != "cks":
        # the contravariant metric: zeros only (its entries are not
        # symmetric bit for bit)
        gc = cen[:, 16:32].reshape(-1, 4, 4)
        for m in (0, 1, 3):
            assert np.all(gc[:, m, 2] == 0.0) and np.all(gc[:, 2, m] == 0.0)
    if kind == "minkowski":
        assert np.array_equal(cen[:, 16:32].reshape(-1, 4, 4), g[: len(cen)])
        assert np.all(cen[:, 32:35] == 1.0)
        assert np.all(face[:, 20:24] == 1.0)
    if kind == "cks":
        # eta + (xi l_m) l_n, from x as the tables' null vectors are
        for x, a, c in zip(*_points(kind)):
            X, Y, Z = x[1:]
            a2 = a * a
            q = (X * X + Y * Y + Z * Z) - a2
            r = max(np.sqrt(0.5 * (q + np.sqrt(q * q + 4.0 * a2 * Z * Z))), 1.0e-15)
            r2 = r * r
            xi = 2.0 * (r2 * r) / (r2 * r2 + a2 * Z * Z)
            l = [1.0, (r * X + a * Y) / (r2 + a2), (r * Y - a * X) / (r2 + a2), Z / r]
            for m in range(4):
                for n in range(4):
                    eta = (-1.0 if m == 0 else 1.0) if m == n else 0.0
                    assert c[4 * m + n] == eta + (xi * l[m]) * l[n]
    # a face is singular exactly where its lapse entry is zero
    assert np.array_equal(face[:, 22] == 0.0, face[:, 23] == 0.0)
