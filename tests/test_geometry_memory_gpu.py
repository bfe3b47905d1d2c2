"""Device memory of a context's geometry tables: at most a full centre and
face table per cell, also for Cartesian Kerr-Schild, whose kernels read xi and
l in the place of gcov."""
import ctypes as C

import pytest

from pangu_amd import abi, configs
from pangu_amd.tasklist import HipRuntime


def _free(hip):
    a, b = C.c_size_t(), C.c_size_t()
    hip.check(hip.h.hipDeviceSynchronize(), "sync")
    hip.check(hip.h.hipMemGetInfo(C.byref(a), C.byref(b)), "hipMemGetInfo")
    return a.value


@pytest.mark.gpu
def test_cartesian_kerr_schild_tables_take_no_more_than_full_ones():
    hip = HipRuntime()
    hip.check(hip.h.hipSetDevice(0), "hipSetDevice")
    d = configs.orszag_tang(16, (1, 1, 1))
    d.update(nx=[96, 96, 96], nb=[1, 1, 1], xmin=[2.3, 2.2, 2.25], xmax=[3.3, 3.2, 3.25], metric=configs.METRIC["cks"],
             a=0.9375)
    L = abi.lib()
    cfg, blocks = abi.config_from(d), abi.blocks_from(d)
    used = []
    for _ in range(2):  # the first call also loads kernels
        before = _free(hip)
        ctx = C.c_void_p()
        assert L.pangu_create(C.byref(cfg), blocks, 1, 0, C.byref(ctx)) == abi.OK
        used.append(before - _free(hip))
        L.pangu_destroy(ctx)
    n = 96 + 8
    rows = abi.CENTRE_NCOMP * n ** 3 + 3 * abi.FACE_NCOMP * (n + 1) * n * n
    other = 64 << 20  # tile and ghost tables, granularity
    assert used[1] <= 8 * rows + other, (used, 8 * rows)
