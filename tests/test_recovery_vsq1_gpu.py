"""The 2D scheme's iterate at v^2 = 1 exactly, where dP/dv^2 is infinite: a
last step that starts there leaves v^2 at 1 and ends in status 4, so the
chainer goes on to 1Dvsq.  States found by bisection on the 29th iterate with
the scheme compiled for the host; each is checked against the oracle's
scheme."""
import numpy as np
import pytest

import oracle_py as O
from helpers import per_comp_l1
from pangu_amd import configs

# D, tau - D, S_i, B^i of the recovery; rho, u, u~ of the guess
STATES = [
    ("0x1.6cedf6e16d644p-4 -0x1.04a5ea077fb62p+13 0x1.5051c322a76fep-1 -0x1.12da517c8f9bbp-1 -0x1.4bbe3ac0e2007p-1",
     "-0x1.89fb241f968efp+5 0x1.31605173d2210p+3 0x1.aab5f7641efa6p+7",
     "0x1.6cedf6e16d644p-4 0x1.18156a28e68edp+3 0x1.66daaeeb0bc9cp+2 -0x1.2544e59431ff3p+2 -0x1.61f8a71d4cf9dp+2"),
    ("0x1.14024274c27b6p+1 -0x1.19ef5d4c6deefp+7 -0x1.c3c462376d685p-2 0x1.b60ff04a33db0p-4 -0x1.6935318347eeap-3",
     "-0x1.3324fd0877fd4p-5 0x1.0cf2a3aec4c14p-5 -0x1.8f18a2b93f2f1p+4",
     "0x1.14024274c27b6p+1 0x1.800c655345304p+2 -0x1.7cd9ea111c722p+0 0x1.714c349d61dd0p-2 -0x1.3081e4828da09p-1"),
    ("0x1.35492fd600b6ep+4 -0x1.6f865071d3c24p+18 -0x1.5e3c37710a526p-9 -0x1.b25e98401362cp-6 0x1.8f9f5b79c91ebp-6",
     "-0x1.eba45a44ba16dp+5 -0x1.dc8f210157dc1p+9 0x1.cc4e87e101b40p+8",
     "0x1.35492fd600b6cp+4 0x1.8b509722e2ebap-7 -0x1.7f050f71ec31ep-13 -0x1.db0796131aadcp-10 0x1.b507b0bc0f14ep-10"),
    ("0x1.662fccefd4064p+6 -0x1.7e2ba307488cdp+6 0x1.8a7acd4acf425p-2 -0x1.22da0493a982fp-4 0x1.6d36c9ffbf97fp-2",
     "-0x1.027c1210f6f25p+2 0x1.7178a92aa4878p+3 -0x1.8ef42daf7c82ap+3",
     "0x1.662fccefd4063p+6 0x1.97c33e935bc7fp+12 0x1.2897d7c0dd561p-1 -0x1.b55bdf330c6e7p-4 0x1.1296e7ac85fcbp-1"),
    ("0x1.1eace0b90cc46p-6 -0x1.1d10fe40a9d21p-1 -0x1.1f437173702d1p-12 0x1.1125299e8a932p-10 0x1.a692426a26081p-10",
     "-0x1.2d7db916ad329p-2 -0x1.4b5b25a5ec285p-2 0x1.0eef334348f1bp+1",
     "0x1.1eace0b90cc45p-6 0x1.5f9028f5a0687p-8 -0x1.fc98bc82df34ep+4 0x1.e399b1ba43663p+6 0x1.76142e3d99d83p+7"),
    ("0x1.681cae15c8d8ep-5 -0x1.79ff63f319aa1p+9 0x1.b8f79ef79569bp-5 0x1.61ec5a212bf6fp-3 -0x1.29c7025fb8054p-3",
     "-0x1.b074de4318a92p+5 -0x1.f6ae6cf47d36dp+2 -0x1.44467d3141836p+4",
     "0x1.681cae15c8d8dp-5 0x1.517d0270e23afp-10 0x1.30c19ec0d4b93p+4 0x1.e932eac17e5b6p+5 -0x1.9b97d4ea7368ep+5"),
    ("0x1.ed1bad7de697dp-5 -0x1.8a746227c733cp-1 -0x1.a2dea8bd8f432p-7 -0x1.9ac90bb6ec26dp-8 0x1.5918fbb06f8ccp-9",
     "-0x1.e3826b2ffadcfp-1 0x1.96aecd81686eap-3 0x1.540c123fab027p+0",
     "0x1.ed1bad7de697dp-5 0x1.5914d8da4306bp-17 -0x1.4738aa820f2fep+2 -0x1.40e7e1f38f163p+1 0x1.0d9729a945af3p+0"),
    ("0x1.0fcb808ae13efp+1 -0x1.bb3d95bb0a41cp+15 -0x1.8509cebac16f8p+10 -0x1.aed406c59ab28p+11 -0x1.84e21af793aedp+14",
     "-0x1.7d8e54fd9d23dp+8 0x1.468d61bedf07ep+5 0x1.2ec61765c6ef7p+5",
     "0x1.0fcb808ae13edp+1 0x1.4992ab9b97343p+8 -0x1.9a08b7527bdebp+3 -0x1.c6144cba185b5p+4 -0x1.99dedf09eeac0p+7"),
]
GAMMA = 5.0 / 3.0


def _state(words):
    U0, U1, p = ([float.fromhex(x) for x in w.split()] for w in words)
    U = np.array(U0 + U1)
    ent = (GAMMA - 1.0) * p[1] * p[0] ** (-GAMMA)
    return U, np.array(p + list(U[5:8]) + [ent])


@pytest.mark.gpu
def test_an_iterate_at_the_speed_of_light_ends_in_status_4():
    from pangu_amd.sim import HipSim
    cfg = dict(configs.orszag_tang(32, (2, 1, 1)), recovery=0)
    sims = [O.OracleSim(cfg), HipSim(cfg)]
    for s in sims:
        s.init()
        s.task("fix_primitive", 0)
        s.task("conservative", 0)
    o, h = sims
    U, P = o.get("cons", 0), o.get("prim", 0)
    eta = np.diag([-1.0, 1.0, 1.0, 1.0])
    cells = []
    for n, words in enumerate(STATES):
        u, p = _state(words)
        assert O.c2p(0, np.append(u, p[8] * u[0]), p, GAMMA, eta, eta)[0] == 4
        cells.append((n % 2, 0, o.s[1] + 2 + 3 * n, o.s[0] + 5))
        b, k, j, i = cells[-1]
        uc = np.append(u, p[8] * u[0])
        uc[1] = u[1] + u[0]
        assert uc[1] - u[0] == u[1]  # the recovery forms tau - D from it
        U[b, :, k, j, i] = uc
        P[b, :, k, j, i] = p
    for s in sims:
        s.set("cons", U, 1)
        s.set("prim", P, 1)
        s.set("flag", np.ones_like(o.get("flag")))
        s.task("recovery", 0, 1)
    shp = (o.nblocks, 1, o.n[2], o.n[1], o.n[0])
    for f in ("flag", "c2p_status", "c2p_iters"):
        assert np.array_equal(o.interior(o.get(f).reshape(shp)), h.interior(h.get(f).reshape(shp))), f
    it = h.get("c2p_iters").reshape(shp)
    assert all(it[b, 0, k, j, i] > 30 for b, k, j, i in cells)  # the later schemes ran
    lp = per_comp_l1(h.interior(h.get("prim", 1)), o.interior(o.get("prim", 1)))
    assert max(lp) <= 1e-12, lp
