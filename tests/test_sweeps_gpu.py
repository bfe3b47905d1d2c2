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
