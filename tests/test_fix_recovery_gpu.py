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
