"""Ghost exchange and physical boundaries on random fields against plain
numpy copies: every packed component count, one to three dimensions, mixed
boundary kinds, blocks no wider than twice their ghost zones.  Copies and
sign changes only, so the comparison is exact."""
import numpy as np
import pytest

from pangu_amd import abi, configs
from pangu_amd.sim import HipSim

PER, OUT, REF = 0, 1, 2


def _cfg(nx, nb, bc, field, heat):
    d = configs.orszag_tang(nx[0], nb)
    d.update(nx=list(nx), nb=list(nb), bc=[list(p) for p in bc], enable_B=field, enable_heating=heat)
    return d


def _blocks(d):
    return [(i, j, k) for k in range(d["nb"][2]) for j in range(d["nb"][1]) for i in range(d["nb"][0])]


def _boundaries(P, d, field):
    """The X1, X2 and X3 passes in turn on every block."""
    for n, loc in enumerate(_blocks(d)):
        a = P[n]
        for dim in range(3):
            ax = 3 - dim
            size = a.shape[ax]
            if size == 1:
                continue
            for side in (0, 1):
                kind = d["bc"][dim][side]
                edge = loc[dim] == (0 if side == 0 else d["nb"][dim] - 1)
                if not edge or kind == PER:
                    continue
                for g in range(4):
                    dst = g if side == 0 else size - 1 - g
                    src = (4 if side == 0 else size - 5) if kind == OUT else (7 - g if side == 0 else size - 8 + g)
                    v = np.take(a, src, axis=ax).copy()
                    if kind == REF:
                        v[2 + dim] *= -1.0
                        if field:
                            v[5 + dim] *= -1.0
                    idx = [slice(None)] * 4
                    idx[ax] = dst
                    a[tuple(idx)] = v


def _exchange(P, d):
    """Ghosts from the neighbours' interiors; physical sides keep theirs."""
    old, locs = P.copy(), _blocks(d)
    n = [s for s in reversed(P.shape[2:])]
    inner = [s - 8 if s > 1 else 1 for s in n]
    for b, loc in enumerate(locs):
        offs = [(-1, 0, 1) if s > 1 else (0,) for s in n]
        for o2 in offs[2]:
            for o1 in offs[1]:
                for o0 in offs[0]:
                    o = (o0, o1, o2)
                    if o == (0, 0, 0):
                        continue
                    nl = []
                    for dim in range(3):
                        q = loc[dim] + o[dim]
                        if not 0 <= q < d["nb"][dim]:
                            q = q % d["nb"][dim] if d["bc"][dim][0] == PER else None
                        nl.append(q)
                    if None in nl:
                        continue
                    nbk = locs.index(tuple(nl))
                    dst, src = [slice(None)], [slice(None)]
                    for dim in (2, 1, 0):
                        if n[dim] == 1:
                            dst.append(slice(0, 1)), src.append(slice(0, 1))
                            continue
                        lo, hi = {-1: (0, 4), 0: (4, 4 + inner[dim]), 1: (4 + inner[dim], n[dim])}[o[dim]]
                        dst.append(slice(lo, hi))
                        src.append(slice(lo - o[dim] * inner[dim], hi - o[dim] * inner[dim]))
                    P[b][tuple(dst)] = old[nbk][tuple(src)]


CASES = [
    ((40, 1, 1), (2, 1, 1), [(OUT, REF), (PER, PER), (PER, PER)]),
    ((18, 10, 1), (2, 2, 1), [(REF, OUT), (PER, PER), (PER, PER)]),
    ((9, 7, 1), (1, 1, 1), [(OUT, OUT), (REF, REF), (PER, PER)]),
    ((10, 8, 12), (2, 2, 2), [(OUT, OUT), (REF, REF), (PER, PER)]),
    ((5, 8, 7), (1, 2, 1), [(REF, REF), (OUT, REF), (REF, OUT)]),
    ((8, 8, 8), (2, 2, 2), [(PER, PER)] * 3),
]


@pytest.mark.gpu
@pytest.mark.parametrize("nx,nb,bc", CASES)
@pytest.mark.parametrize("field,heat", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_ghost_cells_match_plain_copies(nx, nb, bc, field, heat):
    d = _cfg(nx, nb, bc, field, heat)
    h = HipSim(d)
    h.init()
    rng = np.random.default_rng(3)
    P = rng.normal(size=h.get("prim", 0).shape)
    h.set("prim", P, 0)
    ctx, md, st = h.context()
    L = abi.lib()
    assert L.pangu_exchange_ghosts(ctx, md[0], st) == 0
    _exchange(P, d)
    assert np.array_equal(h.get("prim", 0), P)
    assert L.pangu_apply_boundary_conditions(ctx, md[0], st) == 0
    _boundaries(P, d, field)
    assert np.array_equal(h.get("prim", 0), P)
