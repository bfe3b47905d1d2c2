"""The dt reduction on random wave speeds against numpy: meshes whose items
hold 1, 4 and 16 cells per thread, with partial last steps, one block and
many (both lane widths of the final kernel), NaN speeds among them.  The
maximum and minimum are order-free; a dozen IEEE operations remain."""
import ctypes as C

import numpy as np
import pytest

from pangu_amd import abi, configs
from pangu_amd.sim import HipSim

CASES = [
    ((64, 1, 1), (1, 1, 1)),       # one item
    ((500, 300, 1), (1, 1, 1)),    # 586 items of one cell per thread
    ((1500, 700, 1), (1, 1, 1)),   # 1026 items of four cells per thread, part-filled
    ((100, 90, 344), (1, 1, 4)),   # planes of 9000 cells, sixteen per thread
    ((40, 30, 600), (1, 1, 4)),    # planes of 1200 cells, four per thread
    ((30, 30, 1100), (1, 1, 20)),  # four cells per thread, more than 16 blocks
    ((2048, 2050, 1), (1, 1, 1)),  # sixteen cells per thread
]


@pytest.mark.gpu
@pytest.mark.parametrize("nx,nb", CASES)
def test_timestep_estimate_matches_numpy(nx, nb):
    d = configs.orszag_tang(nx[0], nb)
    d.update(nx=list(nx), nb=list(nb), enable_heating=0)
    h = HipSim(d)
    rng = np.random.default_rng(11)
    a = rng.uniform(0.0, 1.0, h.get("alfven").shape)
    a[rng.random(a.shape) < 1e-3] = np.nan
    h.set("alfven", a)
    ctx, md, st = h.context()
    est = (C.c_double * 1)()
    assert abi.lib().pangu_estimate_timestep(ctx, md[0], est, st) == 0
    want = np.inf
    c = h.interior(a)
    for b in range(h.nblocks):
        s = 0.0
        for q in range(3):
            if nx[q] == 1:
                s = s + 1.0 / np.finfo(np.float64).max
                continue
            s = s + 1.0 / (d["cfl"] * (1.0 / nx[q]) / np.nanmax(c[b, q]))
        want = min(want, 1.0 / s)
    # dx comes from the mesh generator, not from 1 / nx: a few units in the last place
    assert abs(est[0] - want) <= 8 * np.finfo(np.float64).eps * want


# blocks and items of a block that give 1, 1, 2, 4, 8, 16 and 32 lanes to a block
MANY_BLOCKS = [
    ((9000, 1, 1), (1500, 1, 1)),
    ((256, 256, 1), (32, 32, 1)),
    ((64, 64, 64), (8, 8, 8)),
    ((48, 48, 48), (6, 6, 6)),
    ((130, 72, 64), (5, 12, 2)),
    ((96, 80, 62), (8, 5, 1)),
    ((640, 640, 1), (5, 5, 1)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("nx,nb", MANY_BLOCKS)
def test_timestep_estimate_of_many_blocks(nx, nb):
    d = configs.orszag_tang(nx[0], nb)
    d.update(nx=list(nx), nb=list(nb), enable_heating=0)
    h = HipSim(d)
    rng = np.random.default_rng(12)
    a = rng.uniform(0.0, 1.0, h.get("alfven").shape)
    a[rng.random(a.shape) < 1e-3] = np.nan
    h.set("alfven", a)
    ctx, md, st = h.context()
    est = (C.c_double * 1)()
    assert abi.lib().pangu_estimate_timestep(ctx, md[0], est, st) == 0
    c = np.nanmax(h.interior(a).reshape(h.nblocks, 3, -1), axis=2)
    want = np.inf
    for b in range(h.nblocks):
        dx = h.block_geom(b)[0][3:]
        q3 = [np.finfo(np.float64).max if nx[q] == 1 else d["cfl"] * dx[q] / c[b, q] for q in range(3)]
        want = min(want, 1.0 / (1.0 / q3[0] + 1.0 / q3[1] + 1.0 / q3[2]))
    assert est[0] == want  # the same IEEE operations
