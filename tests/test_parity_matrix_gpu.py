"""HIP path vs the oracle across the option matrix: every metric, limiter,
Riemann solver, recovery scheme, heating model and semantics switch, on
small meshes (GPU).  One RK2 cycle each, through the task-by-task ABI and
through the fused stage replayed as a hipGraph."""
import numpy as np
import pytest

import oracle_py as O
from helpers import assert_nonfinite_confined, per_comp_l1
from pangu_amd import configs


def _ot_curved(metric, nx, nb, xmin, xmax, **kw):
    """Orszag-Tang data (unit-period fields) on a patch of a curved
    spacetime: exercises the metric tables, connection and floors with a
    smooth, non-stationary state."""
    d = configs.orszag_tang(nx[0], nb)
    d.update(nx=list(nx), xmin=list(xmin), xmax=list(xmax), metric=configs.METRIC[metric],
             a=0.9375, h=0.0, stage_init=0)
    d.update(kw)
    return d


def _torus2d(**kw):
    d = configs.torus2d(64, 32, (2, 2, 1))
    d.update(kw)
    return d


def _torus3d(**kw):
    d = configs.torus3d((32, 16, 16), (2, 2, 2))
    d.update(kw)
    return d


MATRIX = {
    "ot_cks3d_hll_ppm4_kastaun": _ot_curved("cks", (16, 16, 8), (2, 2, 2), (3.0, -0.5, 1.0),
                                            (4.0, 0.5, 1.5), riemann=1, limiter=1, recovery=1),
    "ot_cks3d_laxf_mc_chainer_heat": _ot_curved("cks", (16, 16, 8), (2, 1, 2), (-4.0, 2.0, -0.5),
                                                (-3.0, 3.0, 0.0), riemann=0, limiter=0,
                                                recovery=0, enable_heating=1, heat_model=2),
    # boxes straddling the excision radius r = 1 (inside the horizon)
    "ot_cks3d_excision_kastaun": _ot_curved("cks", (16, 16, 8), (2, 2, 2), (0.3, 0.2, 0.25),
                                            (1.3, 1.2, 0.75), riemann=1, limiter=1, recovery=1),
    "ot_cks3d_excision_chainer": _ot_curved("cks", (16, 16, 8), (2, 2, 2), (0.6, 0.5, 0.3),
                                            (2.6, 2.5, 1.3), riemann=0, limiter=1, recovery=0,
                                            enable_heating=1),
    # x3-independent blocks: tables of one plane, no X3 faces
    "ot_cks2d_hll_ppm4_kastaun": _ot_curved("cks", (36, 28, 1), (2, 2, 1), (2.3, -0.5, 0.4), (3.3, 0.5, 0.9),
                                            riemann=1, limiter=1, recovery=1, enable_heating=1),
    "ot_cks2d_laxf_mc_chainer": _ot_curved("cks", (36, 28, 1), (1, 2, 1), (-3.3, 1.5, 0.4), (-2.3, 2.5, 0.9),
                                           riemann=0, limiter=0, recovery=0),
    "ot_cks2d_ppm4_kastaun_noB": _ot_curved("cks", (36, 28, 1), (2, 1, 1), (2.3, -0.5, 0.4), (3.3, 0.5, 0.9),
                                            limiter=1, recovery=1, enable_B=0),
    "ot_cks2d_hll_mc_onedvsq_noB": _ot_curved("cks", (36, 28, 1), (2, 2, 1), (2.3, -0.5, 0.4), (3.3, 0.5, 0.9),
                                              riemann=1, limiter=0, recovery=2, enable_B=0),
    "ot_bl2d_hll_mc_chainer": _ot_curved("bl", (32, 32, 1), (2, 2, 1), (1.0, -0.5, 0.0),
                                         (2.0, 0.5, 1.0), riemann=1, limiter=0, recovery=0),
    "ot_mks2d_ppm4_onedvsq": _ot_curved("mks", (32, 32, 1), (1, 2, 1), (1.0, -0.5, 0.0),
                                        (2.0, 0.5, 1.0), h=0.3, limiter=1, recovery=2),
    "ot_minkowski_exchange_after_recovery": dict(configs.orszag_tang(32, (2, 2, 1)),
                                                 exchange_after=1),
    "ot_minkowski_zeroed_stage": dict(configs.orszag_tang(32, (2, 1, 1)), stage_init=0),
    "ot_minkowski_noB": dict(configs.orszag_tang(32), enable_B=0),
    "torus2d_mc_hll": _torus2d(limiter=0, riemann=1),
    "torus2d_kastaun": _torus2d(recovery=1),
    "torus2d_onedvsq": _torus2d(recovery=2),
    "torus2d_heat_howes": _torus2d(heat_model=1),
    "torus2d_heat_kawazura": _torus2d(heat_model=2),
    "torus2d_heat_werner": _torus2d(heat_model=3),
    "torus2d_heat_rowan": _torus2d(heat_model=4),
    "torus2d_heat_sharma": _torus2d(heat_model=5, suppress_highb_heat=1,
                                    enforce_positive_dissipation=1),
    "torus2d_heat_nolimit": _torus2d(limit_kel=0),
    "torus2d_noheat": _torus2d(enable_heating=0),
    "torus3d_chainer_laxf_mc": _torus3d(recovery=0, riemann=0, limiter=0),
    # 1-D mesh (two blocks along x1) and blocks of odd sizes whose face rows
    # do not fill whole wavefronts
    "ot_minkowski_1d": dict(configs.orszag_tang(64, (2, 1, 1)), nx=[64, 1, 1]),
    "torus3d_odd_blocks": configs.torus3d((40, 24, 12), (2, 2, 1)),
    "torus3d_exchange_after_recovery": _torus3d(exchange_after=1),
    # dt reduction with a partial last step: 20x30 planes (600 cells, four
    # cells per thread, the third step part-filled) and one 50x30 plane
    # (1500 cells, sixteen per thread, six steps used)
    "torus3d_dt_600_cell_planes": configs.torus3d((40, 30, 8), (2, 1, 1)),
    "torus2d_dt_1500_cell_plane": configs.torus2d(50, 30, (1, 1, 1)),
}


PAIR_CASES = ["ot_minkowski_1d", "torus3d_odd_blocks", "ot_cks3d_laxf_mc_chainer_heat",
              "torus2d_mc_hll", "ot_bl2d_hll_mc_chainer", "ot_cks3d_excision_kastaun"]


def _compare(o, h, label, tol=1e-12):
    for c in (0, 1):
        lp = per_comp_l1(h.interior(h.get("prim", c)), o.interior(o.get("prim", c)))
        lu = per_comp_l1(h.interior(h.get("cons", c)), o.interior(o.get("cons", c)))
        print(label, "container", c, "P", max(lp), "U", max(lu), flush=True)
        assert max(lp) <= tol, (c, lp)
        assert max(lu) <= tol, (c, lu)
    shp = (o.nblocks, 1, o.n[2], o.n[1], o.n[0])
    for f in ("flag_recovery", "c2p_status", "c2p_iters"):
        a = o.interior(o.get(f).reshape(shp))
        b = h.interior(h.get(f).reshape(shp))
        assert np.array_equal(a, b), (f, int((a != b).sum()))
    assert np.array_equal(o.get("mask").reshape(-1), h.get("mask").reshape(-1))
    assert abs(o.dt - h.dt) <= 1e-15 * o.dt


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["tasks", "graph"])
@pytest.mark.parametrize("name", sorted(MATRIX))
def test_matrix_one_cycle(name, mode):
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    print("case", name, mode, flush=True)
    o = O.OracleSim(cfg)
    o.init()
    h = HipSim(cfg)
    h.init()
    assert np.array_equal(o.get("prim", 0), h.get("prim", 0))
    o.step(1)
    h.step(1, mode)
    _compare(o, h, name)
    for s in (o, h):
        assert_nonfinite_confined(s, cfg, name)


# Failed-recovery patterns (block, k, j, i in interior indices) on 16x8x8 blocks.
FAILURES = [
    (0, 2, 3, 5),                                  # isolated
    (0, 2, 5, 8), (0, 2, 5, 9),                    # pair along i
    (1, 3, 2, 2), (1, 3, 2, 3), (1, 3, 3, 2), (1, 3, 3, 3),  # 2x2 cluster
    *[(2, 4, j, 7) for j in range(8)],             # line along j across the block
    (3, 0, 0, 0), (3, 0, 0, 15),                   # block corners (ghost neighbours)
    (4, 1, 4, 4), (4, 2, 4, 4),                    # neighbours in k only
    (5, 5, 6, 1), (5, 5, 7, 2), (5, 5, 6, 3),      # diagonal chain
]


@pytest.mark.gpu
@pytest.mark.parametrize("name", PAIR_CASES)
def test_matrix_pair_flux(name):
    """The two-lanes-per-face flux sweeps (both limiters and solvers, 1-D to
    3-D, polar and excised faces) against the oracle and bit for bit against
    the one-lane sweeps."""
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    o = O.OracleSim(cfg)
    o.init()
    o.step(1)
    runs = []
    for pair in (0, 7):
        h = HipSim(cfg)
        h.init()
        h.set_pair_flux(pair)
        h.step(1, "graph")
        if pair:
            _compare(o, h, name + " pair")
        runs.append((h.get("prim", 0), h.get("cons", 0), h.get("prim", 1), h.get("alfven")))
        h.close()
    for a, b in zip(runs[0], runs[1]):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("name", PAIR_CASES)
def test_matrix_march_flux(name):
    """The marching X2/X3 sweeps (several faces per thread, one
    reconstruction per cell; depths that do and do not divide the face
    counts, both tile orders) against the oracle and bit for bit against
    the one-face sweeps: fields, face fluxes and wave speeds."""
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    o = O.OracleSim(cfg)
    o.init()
    o.step(1)
    runs = []
    for depth, order in ((0, 0), (3, 0), (4, 1), (7, 0), (64, 1)):
        h = HipSim(cfg)
        h.init()
        for d in (2, 3):
            h.set_flux_march(d, depth)
            h.set_tile_order("flux_x%d" % d, order)
        h.step(1, "graph")
        if depth:
            _compare(o, h, name + " march %d" % depth)
        runs.append((depth, [h.get("prim", 0), h.get("cons", 0), h.get("prim", 1), h.get("alfven"),
                             h.get("flux2"), h.get("flux3")]))
        h.close()
    for depth, fields in runs[1:]:
        for a, b in zip(runs[0][1], fields):
            assert np.array_equal(a, b, equal_nan=True), depth


@pytest.mark.gpu
@pytest.mark.parametrize("name", PAIR_CASES + ["torus2d_kastaun"])
def test_matrix_small_tiles(name):
    """Every kernel family in tiles of 128 and of 64 cells (workgroups of
    that size; 1-D to 3-D, both tile orders; the 128-cell run with the
    persistent work-queue recovery) against the oracle and bit for bit
    against 256-cell tiles."""
    from pangu_amd.sim import HipSim, KERNEL_FAMILIES
    cfg = MATRIX[name]
    o = O.OracleSim(cfg)
    o.init()
    o.step(1)
    runs = []
    for cells, order in ((256, 0), (128, 1), (64, 0)):
        h = HipSim(cfg)
        h.init()
        h.set_persistent_recovery(1 if cells == 128 else 0)
        for fam in KERNEL_FAMILIES:
            h.set_tile_size(fam, cells)
            h.set_tile_order(fam, order)
        h.step(1, "graph")
        if cells != 256:
            _compare(o, h, name + " tile %d" % cells)
        runs.append((cells, [h.get("prim", 0), h.get("cons", 0), h.get("prim", 1), h.get("alfven")]))
        h.close()
    for cells, fields in runs[1:]:
        for a, b in zip(runs[0][1], fields):
            assert np.array_equal(a, b, equal_nan=True), cells


@pytest.mark.gpu
def test_fix_recovery_patterns():
    """Recovery failures planted by making D < 0 in chosen cells; the
    averaging fixer must reproduce the serial lexicographic result of
    recovery_fixer.cc, including clusters, lines and block corners."""
    from pangu_amd.sim import HipSim
    cfg = _torus3d(recovery=0)
    sims = [O.OracleSim(cfg), HipSim(cfg)]
    for s in sims:
        s.init()
        s.task("fix_primitive", 0)
        s.task("conservative", 0)
    o, h = sims
    U = o.get("cons", 0)
    P = o.get("prim", 0)
    for b, k, j, i in FAILURES:
        U[b, 0, o.s[2] + k, o.s[1] + j, o.s[0] + i] = -1.0
    for s in sims:
        s.set("cons", U, 1)
        s.set("prim", P, 1)
        s.set("flag", np.ones_like(o.get("flag")))
        s.task("recovery", 0, 1)
    fo, fh = o.interior(o.get("flag")), h.interior(h.get("flag"))
    assert np.array_equal(fo, fh)
    assert int((fo == 0).sum()) >= len(FAILURES)
    for s in sims:
        s.task("fix_recovery", 0, 1)
    lp = per_comp_l1(h.interior(h.get("prim", 1)), o.interior(o.get("prim", 1)))
    print("fix_recovery P", max(lp), flush=True)
    assert max(lp) <= 1e-13
    assert np.array_equal(o.interior(o.get("flag")), h.interior(h.get("flag")))


def _third_stage_states(n, seed=11):
    """States whose recovery reaches the chainer's third scheme and succeeds
    there (invertor.cc:184-198): magnetised flat-space states whose momentum
    is inflated past the energy's reach, with the exact primitives as the
    guess.  2D (scheme_2d.h) and 1Dvsq (scheme_1d_vsq.h) then stop without
    converging (status 101) and 1D (scheme_1d.h:411-568) converges.  Found by
    a seeded search with the oracle's per-scheme solvers; each is checked
    scheme by scheme.  Returns (U as the conserved container holds it,
    guess) pairs and the per-scheme (status, iterations)."""
    gam = 5.0 / 3.0
    eta = np.diag([-1.0, 1.0, 1.0, 1.0])
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(200000):
        p = np.zeros(10)
        p[0] = 10 ** rng.uniform(-3, 1)
        p[1] = p[0] * 10 ** rng.uniform(-6, 1)
        p[2:5] = rng.normal(size=3) * 10 ** rng.uniform(-1, 1.5)
        p[5:8] = rng.normal(size=3) * np.sqrt(p[0]) * 10 ** rng.uniform(-1, 2)
        p[8] = (gam - 1.0) * p[1] * p[0] ** (-gam)
        U = O.flux(gam, p, eta, eta, -1.0, 0)[:9]
        U[2:5] *= 1.0 + 10 ** rng.uniform(-3, 1)
        Uh = U.copy()
        Uh[1] = U[1] - U[0]  # invertor.cc:149-174 with alpha = sqrt|g| = 1
        g = p[:9].copy()
        s1, _, i1 = O.c2p(1, Uh, g, gam, eta, eta)
        if s1 == 0:
            continue
        s0, _, i0 = O.c2p(0, Uh, g, gam, eta, eta)
        s2, _, i2 = O.c2p(2, Uh, g, gam, eta, eta)
        if s0 != 0 and s2 == 0:
            out.append((U, g, ((s0, i0), (s1, i1), (s2, i2))))
            if len(out) == n:
                break
    assert len(out) == n
    return out


@pytest.mark.gpu
def test_chainer_third_stage_succeeds():
    """Cells whose 2D and 1Dvsq recoveries fail and whose 1D recovery
    succeeds, planted in a chainer run on a flat mesh next to D < 0 cells
    that fail all three: status, iteration counts (the sum over the schemes
    tried), flags and recovered fields equal the oracle's."""
    from pangu_amd.sim import HipSim
    cfg = dict(configs.orszag_tang(32, (2, 2, 1)), recovery=0)
    states = _third_stage_states(12)
    sims = [O.OracleSim(cfg), HipSim(cfg)]
    for s in sims:
        s.init()
        s.task("fix_primitive", 0)
        s.task("conservative", 0)
    o, h = sims
    U = o.get("cons", 0)
    P = o.get("prim", 0)
    cells = [(b, 0, j, i) for b in range(4) for j, i in ((2, 3), (9, 12), (14, 0))]
    for (b, k, j, i), (u, g, _) in zip(cells, states):
        at = (b, slice(None), o.s[2] + k, o.s[1] + j, o.s[0] + i)
        U[at] = u
        P[at] = g
    dneg = [(0, 0, 7, 7), (3, 0, 5, 10)]
    for b, k, j, i in dneg:
        U[b, 0, o.s[2] + k, o.s[1] + j, o.s[0] + i] = -1.0
    for s in sims:
        s.set("cons", U, 1)
        s.set("prim", P, 1)
        s.set("flag", np.ones_like(o.get("flag")))
        s.task("recovery", 0, 1)
    shp = (o.nblocks, 1, o.n[2], o.n[1], o.n[0])
    st = {}
    for f in ("flag_recovery", "c2p_status", "c2p_iters"):
        a = o.get(f).reshape(shp)
        b = h.get(f).reshape(shp)
        assert np.array_equal(o.interior(a), h.interior(b)), f
        st[f] = a
    for (b, k, j, i), (_, _, per) in zip(cells, states):
        at = (b, 0, o.s[2] + k, o.s[1] + j, o.s[0] + i)
        assert st["c2p_status"][at] == 0 and st["flag_recovery"][at] == 1.0
        assert st["c2p_iters"][at] == per[0][1] + per[1][1] + per[2][1]
    for b, k, j, i in dneg:
        assert st["c2p_status"][b, 0, o.s[2] + k, o.s[1] + j, o.s[0] + i] != 0
    lp = per_comp_l1(h.interior(h.get("prim", 1)), o.interior(o.get("prim", 1)))
    print("third stage P", max(lp), flush=True)
    assert max(lp) <= 1e-12
    Po, Ph = o.get("prim", 1), h.get("prim", 1)
    for b, k, j, i in cells:
        at = (b, slice(0, 5), o.s[2] + k, o.s[1] + j, o.s[0] + i)
        assert np.allclose(Ph[at], Po[at], rtol=1e-12, atol=0.0)


@pytest.mark.gpu
def test_launch_tuning_leaves_results_unchanged():
    """Tile order, the split of the source kernel and forming the CT face
    fluxes inside the update kernel change only the launch schedule: one
    graph cycle gives bit-identical fields either way."""
    from pangu_amd.sim import HipSim, KERNEL_FAMILIES
    cfg = _torus3d()
    runs = []
    for variant in ("default", "split", "column", "plane", "share", "ct_faces", "split_ct_faces",
                    "pair", "pair_share", "march", "march_column", "tile128", "tile64",
                    "tile64_column", "persistent", "persistent_tile64", "overlap", "separate_update_recovery"):
        h = HipSim(cfg)
        h.init()
        if variant in ("split", "split_ct_faces"):
            h.set_split_source(1)
        if variant in ("ct_faces", "split_ct_faces"):
            h.set_fuse_ct(0)
        if variant in ("share", "pair_share"):
            h.set_share_reconstruction(1)
        if variant in ("pair", "pair_share"):
            h.set_pair_flux(7)
        if variant in ("march", "march_column"):
            h.set_flux_march(2, 5)
            h.set_flux_march(3, 3)
        if variant.startswith("persistent"):
            h.set_persistent_recovery(1)
        if variant == "overlap":
            h.set_overlap_exchange(1)
        if variant == "separate_update_recovery":
            h.set_fuse_update_recovery(0)
        for fam in KERNEL_FAMILIES:
            if variant.startswith("tile"):
                h.set_tile_size(fam, int(variant[4:].split("_")[0]))
            if variant == "persistent_tile64":
                h.set_tile_size(fam, 64)
            if variant in ("column", "march_column", "tile64_column"):
                h.set_tile_order(fam, 1)
            if variant == "plane":
                h.set_tile_order(fam, 0)
        h.step(2, "graph")
        runs.append((variant, h.get("prim", 0), h.get("cons", 0), h.get("prim", 1)))
        h.close()
    for v, P, U, P1 in runs[1:]:
        assert np.array_equal(P, runs[0][1]), v
        assert np.array_equal(U, runs[0][2]), v
        assert np.array_equal(P1, runs[0][3]), v


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ot_minkowski_exchange_after_recovery", "torus2d_kastaun",
                                  "ot_minkowski_1d", "ot_cks3d_hll_ppm4_kastaun"])
def test_fused_ct_is_bit_identical(name):
    """The update kernel's own CT face fluxes (from the edge EMFs) give the
    same bits as writing them with the face kernel first, in 1-D, 2-D and
    3-D."""
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    out = []
    for fuse in (1, 0):
        h = HipSim(cfg)
        h.init()
        h.set_fuse_ct(fuse)
        h.step(3, "graph")
        out.append((h.get("prim", 0), h.get("cons", 0), h.get("prim", 1)))
        h.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ot_minkowski_noB", "torus2d_mc_hll", "torus2d_kastaun",
                                  "ot_cks3d_laxf_mc_chainer_heat", "torus3d_odd_blocks", "ot_minkowski_1d"])
def test_fused_fix_x1_is_bit_identical(name):
    """FixPrimitive + conservative and the X1 sweep in one kernel (halo cells
    fixed twice, the fixed primitives kept in LDS) give the same bits as the
    two kernels: fields, masks, X1 fluxes and wave speeds, for both limiters
    and solvers, with and without a field and K_e."""
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    out = []
    for fuse in (0, 1):
        h = HipSim(cfg)
        h.init()
        h.set_fuse_fix_x1(fuse)
        h.step(3, "graph")
        out.append([h.get(f, c) for f, c in (("prim", 0), ("cons", 0), ("prim", 1), ("mask", 0),
                                              ("flux1", 0), ("alfven", 0))])
        h.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ot_minkowski_noB", "torus2d_mc_hll", "ot_cks3d_laxf_mc_chainer_heat"])
def test_shared_reconstruction_is_bit_identical(name):
    """The X1 sweep with one reconstruction per cell (wavefront shuffle of
    the right interface value) gives the same bits as the per-face sweep,
    for both limiters and both solvers."""
    from pangu_amd.sim import HipSim
    cfg = MATRIX[name]
    out = []
    for share in (0, 1):
        h = HipSim(cfg)
        h.init()
        h.set_share_reconstruction(share)
        h.step(2, "graph")
        out.append((h.get("prim", 0), h.get("cons", 0), h.get("flux1")))
        h.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)
