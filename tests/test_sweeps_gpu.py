"""All sweeps and the ghost exchange in one launch against one launch each
(a tile size of its own for X1 keeps the directions apart): bit-identical,
from one tile per direction to several runs per XCD, one to three
dimensions, uneven meshes in one context."""
import numpy as np
import pytest

from pangu_amd import configs
from pangu_amd.sim import HipSim

CASES = {
    "1d": [dict(configs.orszag_tang(50, (2, 1, 1)), nx=[50, 1, 1])],
    "2d": [configs.orszag_tang(48, (2, 3, 1))],
    "3d_odd": [configs.torus3d((38, 22, 14), (2, 2, 2))],
    "3d_runs": [configs.torus3d((128, 96, 64), (2, 2, 1))],
    "batch": configs.ensemble(seed=3, n_tori=2, n_boxes_each=2, sizes3d=(16,), tori_res=((64, 32), (80, 48))),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_merged_sweeps_are_bit_identical(name):
    runs = []
    for tile in (256, 128):
        h = HipSim(CASES[name] if len(CASES[name]) > 1 else CASES[name][0])
        h.init()
        h.set_tile_size("flux_x1", tile)
        h.step(3, "fused")
        runs.append([h.get(f, c) for f in ("prim", "cons") for c in (0, 1)] + [h.get("alfven")])
    for a, b in zip(*runs):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.gpu
def test_exchange_waits_for_sweeps_of_the_same_primitives():
    """Two handles on one set of primitives, as input and output of a stage:
    the exchange must not refresh the ghosts the sweeps still read (stale on
    purpose here).  Equal to the stage whose input and output are one
    handle."""
    import ctypes as C

    from pangu_amd.tasklist import TaskList
    cfg = configs.orszag_tang(96, (2, 1, 1))
    h = HipSim(cfg)
    h.init()
    P = h.get("prim", 0)
    P[..., :4] *= 1.01  # x1 ghosts
    out = []
    for target in ("1", "dudt"):  # "dudt" has the primitives of "1"
        t = TaskList(cfg)
        t.set("prim", P, "base")
        t.set("prim", P, "1")
        L, m = t.L, t.handle
        t._ok(L.pangu_fix_primitive(t.ctx, m["base"], None), "fix_primitive")
        t._ok(L.pangu_calculate_conservative(t.ctx, m["base"], None), "conservative")
        dt = t.hip.alloc(16)
        t.hip.upload(dt, np.array([1e-4, 0.0]))
        t._ok(L.pangu_stage(t.ctx, m["base"], m["1"], m[target], 0.5, C.cast(C.c_void_p(dt), C.POINTER(C.c_double)),
                            1.0, 0, 0, None), "stage")
        out.append(t.get("prim", "1"))
        t.hip.free(dt)
    assert np.array_equal(out[0], out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("md0,md1", [("mixed", "base"), ("mixed", "1"), ("base", "mixed"), ("1", "mixed")])
@pytest.mark.parametrize("overlap", [-1, 1])
def test_exchange_waits_when_some_primitives_are_shared(md0, md1, overlap):
    """A third container that takes its primitives in turn from two which
    share none: with either of the two it is one container to the exchange.
    Equal to the stage whose sweeps run one by one with the exchange after
    them (an option that keeps it out of their launch)."""
    import ctypes as C

    from pangu_amd import abi
    from pangu_amd.tasklist import TaskList, _table
    cfg = configs.orszag_tang(96, (2, 1, 1))
    h = HipSim(cfg)
    h.init()
    P = h.get("prim", 0)
    P[..., :4] *= 1.01  # x1 ghosts that the exchange would change
    out = []
    for plain in (0, 1):
        t = TaskList(cfg)
        cont = abi.PanguContainer()
        tables = []

        def add(ptrs):
            tables.append(_table(ptrs))
            return C.cast(tables[-1], abi._PPD)

        cont.prim = add([(a, b)[q % 2] for q, (a, b) in enumerate(zip(t.ptr[("prim", "base")], t.ptr[("prim", "1")]))])
        cont.cons = add(t.ptr[("cons", "dudt")])
        for d in range(3):
            cont.flux[d] = add(t.ptr[("flux", "1")][d]) if t.ptr[("flux", "1")][d] else abi._PPD()
        mixed = C.c_int()
        t._ok(t.L.pangu_register_container(t.ctx, C.byref(cont), C.byref(mixed)), "register")
        m = dict(t.handle, mixed=mixed.value)
        assert m["mixed"] > max(m["base"], m["1"])
        t.set("prim", P, "base")
        t.set("prim", P, "1")
        L = t.L
        t._ok(L.pangu_fix_primitive(t.ctx, m[md0], None), "fix_primitive")
        t._ok(L.pangu_calculate_conservative(t.ctx, m[md0], None), "conservative")
        t._ok(L.pangu_set_overlap_exchange(t.ctx, 0 if plain else overlap), "overlap")
        t._ok(L.pangu_set_share_reconstruction(t.ctx, plain), "share")
        dt = t.hip.alloc(16)
        t.hip.upload(dt, np.array([1e-4, 0.0]))
        t._ok(L.pangu_stage(t.ctx, m[md0], m[md0], m[md1], 0.5, C.cast(C.c_void_p(dt), C.POINTER(C.c_double)),
                            1.0, 0, 0, None), "stage")
        out.append([t.get("prim", "base"), t.get("prim", "1")])
        t.hip.free(dt)
        t.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
