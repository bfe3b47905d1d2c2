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
