"""FixRecovery on planes of many tiles against the oracle's serial order:
random failed cells from isolated to dense, several containers in turn (the
per-plane words must be back at zero after each), rows that do not fill whole
tiles, an excised region."""
import numpy as np
import pytest

import oracle_py as O
from helpers import per_comp_l1
from pangu_amd import configs


def _cks():
    d = configs.orszag_tang(16, (2, 2, 2))
    d.update(nx=[24, 24, 16], xmin=[0.3, 0.2, 0.25], xmax=[1.3, 1.2, 0.75], metric=configs.METRIC["cks"], a=0.9375,
             recovery=0, stage_init=0)
    return d


CASES = {
    "ot_130x70": dict(configs.orszag_tang(130, (1, 1, 1)), nx=[130, 70, 1], recovery=0),
    "ot_2x2": dict(configs.orszag_tang(64, (2, 2, 1)), recovery=0),
    "ot_1d": dict(configs.orszag_tang(600, (2, 1, 1)), nx=[600, 1, 1], recovery=0),
    "cks_excised": _cks(),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_fix_recovery_matches_the_serial_order(name):
    from pangu_amd.sim import HipSim
    o, h = O.OracleSim(CASES[name]), HipSim(CASES[name])
    rng = np.random.default_rng(5)
    shp = h.get("prim", 0).shape
    for share in (0.0, 0.003, 0.05, 0.5):
        P = rng.uniform(0.5, 2.0, shp)
        fl = (rng.random((shp[0], 1) + shp[2:]) >= share).astype(float)
        for s in (o, h):
            s.set("prim", P.reshape(o.get("prim", 1).shape), 1)
            s.set("flag", fl.reshape(o.get("flag").shape))
            s.task("fix_recovery", 0, 1)
        a = o.interior(o.get("flag").reshape((shp[0], 1) + shp[2:]))
        b = h.interior(h.get("flag").reshape((shp[0], 1) + shp[2:]))
        assert np.array_equal(a, b), share
        # means of the same neighbours in the same order
        lp = per_comp_l1(h.interior(h.get("prim", 1)), o.interior(o.get("prim", 1)))
        assert max(lp) <= 1e-15, (share, lp)


LONG_ROWS = {
    "2d_1500x70": dict(configs.orszag_tang(64, (1, 1, 1)), nx=[1500, 70, 1], recovery=0),
    "1d_2600": dict(configs.orszag_tang(64, (1, 1, 1)), nx=[2600, 1, 1], recovery=0),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(LONG_ROWS))
def test_rows_longer_than_the_held_steps(name):
    """Bands of more steps than are held at a time (kFixSteps): single pairs,
    pairs at the step limits, dense failures."""
    from pangu_amd.sim import HipSim
    o, h = O.OracleSim(LONG_ROWS[name]), HipSim(LONG_ROWS[name])
    rng = np.random.default_rng(6)
    shp = h.get("prim", 0).shape
    s, e = h.s, h.e

    def pairs(n):
        f = np.ones((shp[0], 1) + shp[2:])
        for _ in range(n):
            i, j = rng.integers(s[0], e[0]), rng.integers(s[1], e[1] + 1)
            f[:, :, s[2], j, i:i + 2] = 0.0
        return f

    edges = np.ones((shp[0], 1) + shp[2:])
    for r in range(s[1], e[1] + 1):  # steps 1023 and 1024 of the first band
        c = s[0] + 1023 - 2 * (r - s[1])
        edges[:, :, s[2], r, c:c + 2] = 0.0
    for fl in (pairs(1), pairs(40), edges, (rng.random((shp[0], 1) + shp[2:]) >= 0.4).astype(float)):
        P = rng.uniform(0.5, 2.0, shp)
        for q in (o, h):
            q.set("prim", P.reshape(o.get("prim", 1).shape), 1)
            q.set("flag", fl.reshape(o.get("flag").shape))
            q.task("fix_recovery", 0, 1)
        assert np.array_equal(o.interior(o.get("flag").reshape(fl.shape)), h.interior(h.get("flag").reshape(fl.shape)))
        lp = per_comp_l1(h.interior(h.get("prim", 1)), o.interior(o.get("prim", 1)))
        assert max(lp) <= 1e-15, lp


@pytest.mark.gpu
def test_a_pair_per_band_costs_little():
    """One pair of failed cells in each band of 64 rows against every cell
    failed: a band then has two steps to take instead of 134 (0.03 of the
    dense time; with every step taken 0.19)."""
    import time

    from pangu_amd import abi, sim
    h = sim.HipSim(dict(configs.orszag_tang(64, (1, 1, 1)), nx=[8, 1024, 1], recovery=0))
    P = np.random.default_rng(7).uniform(0.5, 2.0, h.get("prim", 0).shape)
    h.set("prim", P, 1)
    ctx, md, st = h.context()
    L = abi.lib()
    dense = np.zeros(h.get("flag").shape)
    pair = np.ones_like(dense)
    pair[..., h.s[1] + 30:h.e[1]:64, h.s[0] + 3:h.s[0] + 5] = 0.0
    best = {}
    for name, fl in (("pair", pair), ("dense", dense)):
        for _ in range(10):
            h.set("flag", fl)
            sim.lib().pangu_sim_sync(h._p)
            t0 = time.perf_counter()
            assert L.pangu_fix_recovery(ctx, md[1], st) == 0
            assert sim.lib().pangu_sim_sync(h._p) == 0
            best[name] = min(best.get(name, 1e9), time.perf_counter() - t0)
    assert best["pair"] < 0.125 * best["dense"], best
