"""Performance cases of the GRMHD update path.

Each case is a dict of plain values; prepare() makes what a program holds
before the call (fields on the GPU, the context, a captured cycle), run()
makes one pass through the public entry points and returns whole fields, and
exact() restates the result in plain FP64 numpy where that is affordable.

Four kinds:
  step     the Python driver: HipSim.step in graph mode, then the state read
           back, as a script that watches a small run does;
  cycle    one RK2 cycle of pangu_stage on the caller's own containers, either
           called stage by stage or captured once and replayed ("graph");
  tasks    one RK2 cycle task by task with the host's dt, as a task list
           drives the C ABI;
  layer    one step of the path on its own: the flux sweeps, FixPrimitive
           with the conserved state, or the recovery.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from pangu_amd import abi, configs
from pangu_amd.sim import HipSim

NG = 4
RHO, ENY, UX1, UX2, UX3, BX1, BX2, BX3, ENT, KEL = range(10)


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a script's small 2-D test run: launches and the host path count
        dict(name="ot_64_step", kind="step", problem="ot", nx1=64, nx2=64, cycles=5),
        # the 2-D Orszag-Tang benchmark size, replayed as a production run does
        dict(name="ot_256", kind="cycle", problem="ot", nx1=256, nx2=256, nx3=1, nb1=1, nb2=1, nb3=1, graph=True),
        # the 2-D torus benchmark: curved metric, PPM4, Newton chain, heating
        dict(name="torus2d_512x256", kind="cycle", problem="torus2d", nx1=512, nx2=256, nx3=1, nb1=1, nb2=1, nb3=1,
             graph=True),
        # a small 3-D torus in 8 blocks, stage calls made one by one
        dict(name="torus3d_64x32x32", kind="cycle", problem="torus3d", nx1=64, nx2=32, nx3=32, nb1=2, nb2=2, nb3=2,
             graph=False),
        # the 3-D benchmark run: 32 blocks of 64x64x32
        dict(name="torus3d_256x128x128", kind="cycle", problem="torus3d", nx1=256, nx2=128, nx3=128, nb1=4, nb2=2,
             nb3=4, graph=True),
        # ragged single block at the granularity of a Parthenon task list, with
        # a heating model that evaluates powers and the other limiter
        dict(name="torus3d_75x45x27_tasks", kind="tasks", problem="torus3d", nx1=75, nx2=45, nx3=27, nb1=1, nb2=1,
             nb3=1, limiter="mc", heat="howes"),
        # an ensemble of uneven meshes in one context
        dict(name="ensemble_24", kind="cycle", problem="ensemble", tori=12, boxes=4, meshes=0, graph=True),
        # static refinement in Cartesian Kerr-Schild: 3-D geometry tables,
        # hydrodynamic, ghost cells across levels
        dict(name="refined_cks", kind="cycle", problem="cks", nx1=32, nb1=4, levels=2, field=False, graph=True),
        # the three flux sweeps alone, curved metric, PPM4 + HLL, four blocks
        dict(name="fluxes_mks_96x64x32", kind="layer", layer="fluxes", metric="mks", limiter="ppm4", riemann="hll",
             nx1=96, nx2=64, nx3=32, nb1=2, nb2=2, nb3=1),
        # floors and the conserved state, whole ghosted blocks
        dict(name="fix_cons_mks_128x64x64", kind="layer", layer="fix_cons", metric="mks", nx1=128, nx2=64, nx3=64,
             nb1=2, nb2=1, nb3=2),
        # false-position recovery and heating of magnetised states
        dict(name="recovery_robuster_128x64x64", kind="layer", layer="recovery", metric="mks", recovery="robuster",
             nx1=128, nx2=64, nx3=64, nb1=2, nb2=1, nb3=2),
        # the Newton chain on a ragged 2-D plane in flat space
        dict(name="recovery_chainer_301x199", kind="layer", layer="recovery", metric="minkowski", recovery="chainer",
             nx1=301, nx2=199, nx3=1, nb1=1, nb2=1, nb3=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(("step", "ot", "torus2d", "torus3d", "torus3d", "tasks", "ensemble", "cks", "fluxes", "fix_cons",
                       "recovery", "recovery"))
    if what == "step":
        return dict(kind="step", problem="ot", nx1=_log_int(rng, 24, 160), nx2=_log_int(rng, 24, 160),
                    cycles=rng.randint(1, 12))
    if what in ("ot", "torus2d"):
        b1, b2 = rng.choice((1, 1, 2)), rng.choice((1, 2, 3))
        return dict(kind="cycle", problem=what, nx1=b1 * _log_int(rng, 24, 512), nx2=b2 * _log_int(rng, 20, 256), nx3=1,
                    nb1=b1, nb2=b2, nb3=1, graph=rng.random() < 0.7)
    if what == "torus3d":
        b1, b2, b3 = rng.choice((1, 2, 4)), rng.choice((1, 2)), rng.choice((1, 2, 4))
        return dict(kind="cycle", problem="torus3d", nx1=b1 * _log_int(rng, 17, 64), nx2=b2 * _log_int(rng, 16, 64),
                    nx3=b3 * _log_int(rng, 12, 32), nb1=b1, nb2=b2, nb3=b3, graph=rng.random() < 0.7)
    if what == "tasks":
        return dict(kind="tasks", problem="torus3d", nx1=_log_int(rng, 20, 96), nx2=_log_int(rng, 16, 64),
                    nx3=_log_int(rng, 9, 40), nb1=1, nb2=1, nb3=1, limiter=rng.choice(("mc", "ppm4")),
                    heat=rng.choice(("constant", "howes", "kawazura", "werner", "rowan", "sharma")))
    if what == "ensemble":
        return dict(kind="cycle", problem="ensemble", tori=rng.randint(2, 16), boxes=rng.randint(1, 5),
                    meshes=rng.randrange(1000), graph=True)
    if what == "cks":
        return dict(kind="cycle", problem="cks", nx1=4 * rng.choice((6, 8, 10, 12)), nb1=4, levels=rng.choice((1, 2)),
                    field=rng.random() < 0.5, graph=rng.random() < 0.7)
    metric = rng.choice(("mks", "mks", "minkowski"))
    d = dict(kind="layer", layer=what, metric=metric)
    if what == "fluxes":
        d.update(limiter=rng.choice(("mc", "ppm4")), riemann=rng.choice(("laxf", "hll")))
    if what == "recovery":
        d.update(recovery=rng.choice(("robuster", "chainer")))
    b1, b2 = rng.choice((1, 2)), rng.choice((1, 2))
    if rng.random() < 0.5:
        d.update(nx1=b1 * _log_int(rng, 33, 320), nx2=b2 * _log_int(rng, 17, 160), nx3=1, nb1=b1, nb2=b2, nb3=1)
    else:
        d.update(nx1=b1 * _log_int(rng, 17, 64), nx2=b2 * _log_int(rng, 12, 48), nx3=_log_int(rng, 9, 40), nb1=b1, nb2=b2,
                 nb3=1)
    return d


# ----------------------------------------------------------- configurations
def _configs(case, seed):
    """Run configuration(s) of a case (pangu_amd.configs dicts)."""
    if case["kind"] == "layer":
        d = configs.torus3d()
        d.update(nx=[case["nx1"], case["nx2"], case["nx3"]], nb=[case["nb1"], case["nb2"], case["nb3"]],
                 metric=configs.METRIC[case["metric"]], limiter=configs.LIMITER[case.get("limiter", "ppm4")],
                 riemann=configs.RIEMANN[case.get("riemann", "hll")],
                 recovery=configs.RECOVERY[case.get("recovery", "robuster")], density_floor=1e-4, energy_floor=1e-6)
        if case["metric"] == "minkowski":
            d.update(xmin=[0.0, 0.0, 0.0], xmax=[1.0, 1.0, 1.0])
        return d
    p = case["problem"]
    if p == "ot":
        d = configs.orszag_tang(case["nx1"], (case.get("nb1", 1), case.get("nb2", 1), 1))
        d["nx"] = [case["nx1"], case["nx2"], 1]
        return d
    if p == "torus2d":
        d = configs.torus2d(case["nx1"], case["nx2"], (case["nb1"], case["nb2"], 1))
    elif p == "torus3d":
        d = configs.torus3d((case["nx1"], case["nx2"], case["nx3"]), (case["nb1"], case["nb2"], case["nb3"]))
    elif p == "cks":
        d = configs.fm_torus_cks(case["nx1"], case["nb1"], case["levels"], enable_B=int(case["field"]))
    else:
        # the meshes are the case's; fields and perturbations the seed's
        rng = random.Random(seed)
        out = configs.ensemble(seed=case["meshes"], n_tori=case["tori"], n_boxes_each=case["boxes"], sizes3d=(16, 32),
                               tori_res=((128, 64), (256, 128), (192, 96)))
        for d in out:
            d.update(seed=rng.randrange(1 << 62), beta=math.exp(rng.uniform(math.log(30.0), math.log(300.0))))
        return out
    d["seed"] = seed
    if "limiter" in case:
        d["limiter"] = configs.LIMITER[case["limiter"]]
    if "heat" in case:
        d["heat_model"] = abi.HEAT[case["heat"]]
    return d


# ------------------------------------------------------------- GPU state
def _table(ptrs, ctype=C.c_double):
    t = (C.POINTER(ctype) * len(ptrs))()
    C.memmove(t, (C.c_uint64 * len(ptrs))(*ptrs), 8 * len(ptrs))
    return t


class Fields:
    """A simulation's context with containers of the caller's own: one torch
    tensor per field, laid out [block][component][k][j][i]."""

    def __init__(self, cfg, iters=True):
        self.sim = HipSim(cfg)
        self.cfg = self.sim.cfg
        self.L = abi.lib()
        self.ctx = self.sim.context()[0]
        self.cells = [s[0] * s[1] * s[2] for s in self.sim.shapes]
        self.total = sum(self.cells)
        self.np = 6 + (3 if self.cfg["enable_B"] else 0) + (1 if self.cfg["enable_heating"] else 0)
        self.ndim = 3 if max(s[2] for s in self.sim.shapes) > 1 else 2
        self.t, self._keep = {}, []
        flux = [self._new(f"flux{d + 1}", self.np) for d in range(self.ndim)]
        self.h = {}
        for name in ("base", "1", "dudt"):
            c = abi.PanguContainer()
            c.prim = self._new("prim1" if name == "dudt" else "prim0" if name == "base" else "prim1", self.np)
            c.cons = self._new({"base": "cons0", "1": "cons1", "dudt": "dudt"}[name], self.np)
            for d in range(3):
                c.flux[d] = flux[d] if d < self.ndim and name != "dudt" else abi._PPD()
            h = C.c_int()
            self.ok(self.L.pangu_register_container(self.ctx, C.byref(c), C.byref(h)))
            self.h[name] = h.value
        sh = abi.PanguShared()
        sh.alfven, sh.emf = self._new("alfven", 3), self._new("emf", 3)
        sh.flag = self._new("flag", 1)
        sh.mask = self._new("mask", 1, torch.uint8, C.c_uint8)
        sh.c2p_status = self._new("status", 1, torch.int32, C.c_int32)
        if iters:
            sh.c2p_iters = self._new("iters", 1, torch.int32, C.c_int32)
        self.ok(self.L.pangu_register_shared(self.ctx, C.byref(sh)))
        self.t["flag"].fill_(1.0)
        state = []
        for m in range(self.sim.nmesh):
            dt, time = self.sim.mesh_state(m)[:2]
            state += [dt, time]
        self.t["dt"] = torch.tensor(state, dtype=torch.float64, device="cuda")
        self.graph = None

    def _new(self, name, ncomp, dtype=torch.float64, ctype=C.c_double):
        if name not in self.t:
            self.t[name] = torch.zeros(self.total * ncomp, dtype=dtype, device="cuda")
        a, ptrs, off = self.t[name], [], 0
        for cells in self.cells:
            ptrs += [a.data_ptr() + (off * ncomp + q * cells) * a.element_size() for q in range(ncomp)]
            off += cells
        tab = _table(ptrs, ctype)
        self._keep.append(tab)
        return C.cast(tab, C.POINTER(C.POINTER(ctype)))

    def ok(self, r):
        if r != 0:
            raise RuntimeError(f"pangu call failed ({r}): {self.L.pangu_last_error(self.ctx).decode()}")

    def upload(self, name, arr):
        self.t[name].copy_(torch.from_numpy(np.ascontiguousarray(arr, dtype=np.float64).reshape(-1)))

    def cycle(self):
        """One RK2 cycle with the dt on the device."""
        L, x, h, c = self.L, self.ctx, self.h, self.cfg
        st = torch.cuda.current_stream().cuda_stream
        dt = C.cast(self.t["dt"].data_ptr(), C.POINTER(C.c_double))
        self.ok(L.pangu_stage(x, h["base"], h["base"], h["1"], 0.5, dt, c["dt_factor"], 0, c["exchange_after"], st))
        self.ok(L.pangu_stage(x, h["base"], h["1"], h["base"], 1.0, dt, c["dt_factor"], 1, c["exchange_after"], st))

    def cycle_tasks(self):
        """One RK2 cycle at task granularity with the host's dt."""
        L, x, c = self.L, self.ctx, self.cfg
        s = torch.cuda.current_stream().cuda_stream
        for c0, c1, beta in ((self.h["base"], self.h["1"], 0.5), (self.h["1"], self.h["base"], 1.0)):
            bdt = beta * self.dt
            self.ok(L.pangu_fix_primitive(x, c0, s))
            self.ok(L.pangu_calculate_conservative(x, c0, s))
            self.ok(L.pangu_calculate_fluxes(x, c0, s))
            self.ok(L.pangu_constrained_transport(x, c0, s))
            self.ok(L.pangu_flux_divergence(x, c0, self.h["dudt"], s))
            self.ok(L.pangu_update_independent(x, self.h["base"], self.h["dudt"], bdt, c1, s))
            self.ok(L.pangu_exchange_ghosts(x, c1, s))
            self.ok(L.pangu_add_geometric_source(x, c1, bdt, s))
            self.ok(L.pangu_recovery(x, c1, s))
            self.ok(L.pangu_apply_electron_heating(x, c1, s))
            self.ok(L.pangu_apply_boundary_conditions(x, c1, s))
        est = (C.c_double * 1)()
        self.ok(L.pangu_estimate_timestep(x, c1, est, s))
        self.dt = min(c["dt_factor"] * self.dt, est[0])


def prepare(case, seed):
    cfg = _configs(case, seed)
    if case["kind"] == "step":
        sim = HipSim(cfg)
        p = _ot_state(case, seed)
        sim.set("prim", p, 0)
        sim.set("prim", p, 1)
        return dict(case=case, sim=sim)
    if case["kind"] == "layer":
        f = Fields(cfg, iters=False)
        p, geo = _layer_state(case, seed)
        if case["layer"] == "recovery":
            f.upload("cons0", _conserved(p, geo, cfg["gamma"]))
            f.upload("prim0", _guess(p, seed))
        else:
            f.upload("prim0", p)
    else:
        f = Fields(cfg)
        if case["problem"] == "ot":
            f.upload("prim0", _ot_state(case, seed))
        else:
            f.sim.init()
            f.upload("prim0", f.sim.get("prim", 0))
        if f.cfg["stage_init"] == 1:
            f.t["prim1"].copy_(f.t["prim0"])
        f.dt = f.cfg["dt_init"]
        if case.get("graph"):
            torch.cuda.synchronize()
            f.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(f.graph):
                f.cycle()
    torch.cuda.synchronize()
    return dict(case=case, fields=f)


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        sim = state["sim"]
        sim.step(case["cycles"], "graph")
        return [sim.get("prim", 0), sim.dt]
    f = state["fields"]
    t = f.t
    if case["kind"] == "cycle":
        if f.graph:
            f.graph.replay()
        else:
            f.cycle()
        if case["problem"] == "cks":
            # the conserved state of excised cells is not evolved and may be
            # non-finite; the primitives carry the run
            return [t["prim0"], t["prim1"], t["dt"]]
        return [t["prim0"], t["cons0"], t["prim1"], t["cons1"], t["dt"]]
    if case["kind"] == "tasks":
        f.cycle_tasks()
        return [t["prim0"], t["cons0"], t["prim1"], t["cons1"], f.dt]
    s = torch.cuda.current_stream().cuda_stream
    h = f.h["base"]
    if case["layer"] == "fluxes":
        f.ok(f.L.pangu_calculate_fluxes(f.ctx, h, s))
        return [t[f"flux{d + 1}"] for d in range(f.ndim)] + [t["alfven"]]
    if case["layer"] == "fix_cons":
        f.ok(f.L.pangu_fix_primitive(f.ctx, h, s))
        f.ok(f.L.pangu_calculate_conservative(f.ctx, h, s))
        return [t["prim0"], t["cons0"], t["mask"]]
    f.ok(f.L.pangu_recovery(f.ctx, h, s))
    f.ok(f.L.pangu_apply_electron_heating(f.ctx, h, s))
    return [t["prim0"], t["status"]]


def _zones(case):
    if case.get("problem") == "ensemble":
        # mean torus of the three resolutions, boxes of 16^3 and 32^3
        return case["tori"] * (128 * 64 + 256 * 128 + 192 * 96) // 3 + case["boxes"] * (16 ** 3 + 32 ** 3)
    if case.get("problem") == "cks":
        # blocks of (nx1 / nb1)^3 cells: half of the root blocks per
        # direction are refined at every level (56 stay of 64)
        return (case["nx1"] // case["nb1"]) ** 3 * (56 * case["levels"] + 64)
    return case["nx1"] * case["nx2"] * case.get("nx3", 1)


def work(case):
    """Bytes: every input read and every output written once (a stage reads P
    and the initial U and writes U and P).  Operations: the tabulated-geometry
    algorithm's adds, multiplies, divisions and roots per zone."""
    n = _zones(case)
    p = case.get("problem")
    nc = 9 if p == "ot" or case.get("field") else 6 if p == "cks" else 10
    dim = 3 if case.get("nx3", 1) > 1 or p == "cks" else 2
    sweep = 750 if p == "ot" else 1100 if p == "cks" else 1450
    if case["kind"] == "layer":
        if case["layer"] == "fluxes":
            return {"bytes": 8 * n * (nc + dim * (nc + 1)), "flops": 1450 * dim * n}
        if case["layer"] == "fix_cons":
            return {"bytes": 8 * n * 3 * nc, "flops": 700 * n}
        return {"bytes": 8 * n * 2 * nc, "flops": 800 * n}
    cycles = case.get("cycles", 1)
    return {"bytes": cycles * n * 2 * 8 * 4 * nc, "flops": cycles * n * 2 * (sweep * dim + 1800)}


def tolerance(case):
    """About four times what the outputs move by when every input moves by up
    to one unit in the last place (5e-16 for the sweeps and the conserved
    state, 3e-14 for a torus cycle).  The false-position recovery stops at a
    step of 1e-10, which leaves its roots within about 2e-12."""
    if case["kind"] == "layer":
        return {"rel": 1e-11 if case["layer"] == "recovery" else 5e-15, "differ": 1e-4}
    return {"rel": 1e-13 if case["problem"] == "ot" else 1e-12}


# ------------------------------------------------- inputs (host, FP64)
def _blocks(case):
    """(k, j, i) slices of the mesh's interior held by each block, x1 fastest."""
    nb = [case.get("nb1", 1), case.get("nb2", 1), case.get("nb3", 1)]
    nx = [case["nx1"], case["nx2"], case.get("nx3", 1)]
    n = [nx[d] // nb[d] for d in range(3)]
    for k in range(nb[2]):
        for j in range(nb[1]):
            for i in range(nb[0]):
                yield (k * n[2], (k + 1) * n[2]), (j * n[1], (j + 1) * n[1]), (i * n[0], (i + 1) * n[0])


def _split(case, arr, mode="wrap"):
    """Ghosted blocks (block, comp, k, j, i) of a whole-mesh array."""
    g = [(0, 0)] + [(NG, NG) if n > 1 else (0, 0) for n in arr.shape[1:]]
    a = np.pad(arr, g, mode=mode)
    out = []
    for (k0, k1), (j0, j1), (i0, i1) in _blocks(case):
        out.append(a[:, k0:k1 + 2 * g[1][0], j0:j1 + 2 * g[2][0], i0:i1 + 2 * g[3][0]])
    return np.ascontiguousarray(np.stack(out))


def _ot_state(case, seed):
    """Orszag-Tang vortex on the unit box, phases and a 1 % density noise from
    the seed."""
    rng = np.random.default_rng(seed)
    n1, n2 = case["nx1"], case["nx2"]
    x = ((np.arange(n1) + 0.5) / n1)[None, :]
    y = ((np.arange(n2) + 0.5) / n2)[:, None]
    one = np.ones((n2, n1))
    ph = rng.uniform(0.0, 2.0 * math.pi, 4)
    gamma = 5.0 / 3.0
    rho = 25.0 / (36.0 * math.pi) * (1.0 + 0.01 * rng.uniform(-1.0, 1.0, (n2, n1)))
    pr = 5.0 / (12.0 * math.pi) * one
    v1, v2 = -0.5 * np.sin(2 * math.pi * y + ph[0]) * one, 0.5 * np.sin(2 * math.pi * x + ph[1]) * one
    lor = 1.0 / np.sqrt(1.0 - v1 * v1 - v2 * v2)
    b0 = 1.0 / math.sqrt(4.0 * math.pi)
    p = np.zeros((9, 1, n2, n1))
    p[RHO, 0], p[ENY, 0] = rho, pr / (gamma - 1.0)
    p[UX1, 0], p[UX2, 0] = lor * v1, lor * v2
    p[BX1, 0], p[BX2, 0] = -b0 * np.sin(2 * math.pi * y + ph[2]) * one, b0 * np.sin(4 * math.pi * x + ph[3]) * one
    p[8, 0] = pr * rho ** -gamma
    return _split(case, p)


def _layer_state(case, seed):
    """Magnetised states over the range a torus run meets: density over three
    decades, u / rho from 1e-3 to 1, magnetisation 1e-4 to 3, velocities up to
    a Lorentz factor of about two; smooth waves with cell noise.  Returns the
    primitives (block, comp, k, j, i) and the centre geometry of each block."""
    rng = np.random.default_rng(seed)
    n = (case["nx3"], case["nx2"], case["nx1"])
    ax = [np.linspace(0.0, 2.0 * math.pi, m, endpoint=False) for m in n]
    K, J, I = np.meshgrid(*ax, indexing="ij")

    def wave(amp, noise):
        f = np.zeros(n)
        for _ in range(3):
            m = rng.integers(0, 4, 3)
            f += np.sin(m[0] * K + m[1] * J + m[2] * I + rng.uniform(0, 2 * math.pi))
        return amp * f / 3.0 + noise * rng.uniform(-1.0, 1.0, n)

    cfg = _configs(case, seed)
    geo = [_centre_geometry(case, cfg, b) for b in _blocks(case)]
    p = np.zeros((10, *n))
    p[RHO] = np.exp(wave(3.0, 0.1) - 2.0)
    p[ENY] = p[RHO] * np.exp(wave(3.0, 0.1) - 3.0)
    vel = [wave(0.6, 0.02) for _ in range(3)]
    sig = np.exp(wave(4.0, 0.1) - 4.0)
    dirs = [wave(1.0, 0.05) + 1e-3 for _ in range(3)]
    norm = np.sqrt(sum(d * d for d in dirs))
    for d in range(3):
        p[UX1 + d] = vel[d]
        p[BX1 + d] = dirs[d] / norm * np.sqrt(sig * p[RHO])
    gamma = cfg["gamma"]
    p[ENT] = (gamma - 1.0) * p[ENY] * p[RHO] ** -gamma
    p[KEL] = 0.1 * p[ENT] * np.exp(wave(0.5, 0.05))
    p = _split(case, p)
    for b, g in enumerate(geo):
        # components in the local orthonormal scale of the metric
        for d in range(3):
            s = np.sqrt(np.abs(g["g"][d + 1, d + 1]))
            p[b, UX1 + d] /= s
            p[b, BX1 + d] /= s
    return p, geo


def _guess(p, seed):
    """Previous primitives of a recovery: a few per cent off, B stale, the
    entropy kept."""
    rng = np.random.default_rng(seed + 1)
    q = p * (1.0 + 0.03 * rng.uniform(-1.0, 1.0, p.shape))
    q[:, ENT:] = p[:, ENT:]
    return q


# ------------------------------------------- the path in plain numpy (FP64)
def _axis(cfg, d, lo, n, face):
    """Cell centres (or lower faces) of a block's ghosted axis."""
    nx, x0, x1 = cfg["nx"][d], cfg["xmin"][d], cfg["xmax"][d]
    dx = (x1 - x0) / nx
    g = NG if nx > 1 else 0
    i = np.arange(lo - g, lo + n + g + (1 if face else 0))
    return x0 + (i + (0.0 if face else 0.5)) * dx


def _metric(metric, x1, x2, cfg):
    """Code-basis metric: flat, or Kerr-Schild carried to x1 = ln r and the
    theta map by a central difference of step 1e-5."""
    x1, x2 = np.broadcast_arrays(x1, x2)
    g = np.zeros((4, 4, *x1.shape))
    if metric == "minkowski":
        for m in range(4):
            g[m, m] = -1.0 if m == 0 else 1.0
        return g
    a, h, e = cfg["a"], cfg["h"], 1e-5

    def theta(x):
        return 0.5 * math.pi * (x + 1.0) + 0.5 * h * np.sin(math.pi * (x + 1.0))

    r, th = np.exp(x1), theta(x2)
    j1 = (np.exp(x1 + e) - np.exp(x1 - e)) / ((x1 + e) - (x1 - e))
    j2 = (theta(x2 + e) - theta(x2 - e)) / ((x2 + e) - (x2 - e))
    c, s2 = np.cos(th), np.sin(th) ** 2
    sig = r * r + a * a * c * c
    z = 2.0 * r / sig
    g[0, 0], g[0, 1], g[0, 3] = -1.0 + z, z * j1, -z * a * s2
    g[1, 1], g[1, 3] = (1.0 + z) * j1 * j1, -a * (1.0 + z) * s2 * j1
    g[2, 2] = sig * j2 * j2
    g[3, 3] = s2 * (sig + a * a * s2 * (1.0 + z))
    g[1, 0], g[3, 0], g[3, 1] = g[0, 1], g[0, 3], g[1, 3]
    return g


def _geometry(metric, x1, x2, cfg):
    """Metric, its inverse, sqrt|g|, and whether it is regular, on (j, i)."""
    g = _metric(metric, x1[None, :], x2[:, None], cfg)
    m = np.moveaxis(g, (0, 1), (-2, -1))
    det = np.linalg.det(m)
    ok = g[2, 2] * g[3, 3] != 0.0
    inv = np.zeros_like(m)
    inv[ok] = np.linalg.inv(m[ok])
    return dict(g=g[:, :, None], gi=np.moveaxis(inv, (-2, -1), (0, 1))[:, :, None], sg=np.sqrt(np.abs(det))[None], ok=ok[None],
                r=np.exp(x1)[None, None, :] if metric == "mks" else np.ones((1, 1, len(x1))))


def _centre_geometry(case, cfg, block):
    _, (j0, j1), (i0, i1) = block
    return _geometry(case.get("metric", "minkowski"), _axis(cfg, 0, i0, i1 - i0, False), _axis(cfg, 1, j0, j1 - j0, False), cfg)


def _state(p, G):
    """u^mu, u_mu, b^mu, b_mu, b^2."""
    g, gi = G["g"], G["gi"]
    with np.errstate(divide="ignore", invalid="ignore"):
        alpha = 1.0 / np.sqrt(-gi[0, 0])
        v = [p[UX1], p[UX2], p[UX3]]
        sq = sum(g[a + 1, b + 1] * v[a] * v[b] for a in range(3) for b in range(3))
        u0 = np.sqrt(1.0 + sq) / alpha
        u = [u0] + [v[a] - u0 * gi[0, a + 1] * alpha * alpha for a in range(3)]
        ul = [sum(g[m, k] * u[k] for k in range(4)) for m in range(4)]
        B = [p[BX1], p[BX2], p[BX3]]
        b0 = sum(B[a] * ul[a + 1] for a in range(3))
        b = [b0] + [(B[a] + b0 * u[a + 1]) / u0 for a in range(3)]
        bl = [sum(g[m, k] * b[k] for k in range(4)) for m in range(4)]
        return u, ul, b, bl, sum(b[m] * bl[m] for m in range(4))


def _flux(p, S, sg, d, gamma):
    """sqrt|g| times the conserved vector (d = 0) or its flux along d."""
    u, ul, b, bl, bsq = S
    pg = (gamma - 1.0) * p[ENY]
    etot, ptot = p[RHO] + gamma * p[ENY] + bsq, pg + 0.5 * bsq
    T = [etot * u[d] * ul[m] + (ptot if m == d else 0.0) - b[d] * bl[m] for m in range(4)]
    mass = p[RHO] * u[d]
    f = [mass, T[0] + mass, T[1], T[2], T[3]] + [b[a] * u[d] - b[d] * u[a] for a in (1, 2, 3)]
    f += [p[q] * mass for q in range(8, len(p))]
    return np.stack([sg * c for c in f])


def _conserved(p, geo, gamma):
    """U of the interior cells (block, comp, k, j, i); zero in the ghosts."""
    out = np.zeros_like(p)
    for b, G in enumerate(geo):
        out[b] = _flux(p[b], _state(p[b], G), G["sg"], 0, gamma)
    keep = np.zeros(p.shape[2:], dtype=bool)
    keep[_interior(p.shape[2:])] = True
    return np.where(keep, out, 0.0)


def _interior(n, lo=0, hi=0):
    return tuple(slice(NG + lo, m - NG + hi) if m > 1 else slice(None) for m in n)


def _fixed(p, G, cfg):
    """FixPrimitive: floors, the Lorentz cap and the entropies; mask bits."""
    p = p.copy()
    r = np.maximum(G["r"], 1.0)
    smax, gamma = cfg["sigma_max"], cfg["gamma"]
    rfl = np.maximum(cfg["density_floor"] * r ** cfg["density_floor_pow"], p[ENY] / smax)
    efl = np.broadcast_to(cfg["energy_floor"] * r ** cfg["energy_floor_pow"], p[ENY].shape)
    bsq = _state(p, G)[4]
    hot = bsq / p[RHO] > smax
    rfl = np.where(hot, bsq / smax, rfl)
    low, cold = p[RHO] < rfl, p[ENY] < efl
    before = np.maximum(p[RHO], 1e-20)
    p[RHO] = np.where(low, rfl, p[RHO])
    p[ENY] = np.where(cold, efl, p[ENY])
    uu = sum(G["g"][a + 1, b + 1] * p[UX1 + a] * p[UX1 + b] for a in range(3) for b in range(3))
    top = cfg["lorentz_max"] ** 2 - 1.0
    fast = uu > top
    for a in range(3):
        p[UX1 + a] = np.where(fast, p[UX1 + a] * np.sqrt(top / np.maximum(uu, 1e-20)), p[UX1 + a])
    p[8] = (gamma - 1.0) * p[ENY] * p[RHO] ** -gamma
    if len(p) > KEL:
        kel = p[KEL] * (np.maximum(p[RHO], 1e-20) / before) ** -gamma
        kel = np.maximum(0.0, np.minimum(kel, p[8]))
        p[KEL] = np.maximum(p[8] / (1.0 + cfg["ratio_max"]), np.minimum(kel, p[8] / (1.0 + cfg["ratio_min"])))
    return p, (8 * hot + low + 2 * cold + 4 * fast).astype(np.uint8)


def _shift(a, axis, n):
    return np.roll(a, -n, axis=axis)


def _faces(p, axis, limiter):
    """Left and right states of the lower face of every cell along axis."""
    q = [_shift(p, axis, n) for n in (-2, -1, 0, 1, 2)]
    if limiter == "mc":
        a, b, c = 2.0 * (q[2] - q[1]), 0.5 * (q[3] - q[1]), 2.0 * (q[3] - q[2])
        up = np.minimum(np.minimum(a, b), c) * ((a > 0) & (b > 0) & (c > 0))
        s = up + np.maximum(np.maximum(a, b), c) * ((a < 0) & (b < 0) & (c < 0))
        lo, hi = q[2] - 0.5 * s, q[2] + 0.5 * s
    else:
        def edge(m2, m1, z, p1):
            e = (7.0 * (m1 + z) - (m2 + p1)) / 12.0
            return np.minimum(np.maximum(e, np.minimum(m1, z)), np.maximum(m1, z))

        lo, hi = edge(q[0], q[1], q[2], q[3]), edge(q[1], q[2], q[3], q[4])
        c, d = hi - q[2], lo - q[2]
        flat = c * d >= 0.0
        hi2 = np.where(np.abs(c) >= 2.0 * np.abs(d), q[2] - 2.0 * d, hi)
        lo2 = np.where(np.abs(d) >= 2.0 * np.abs(c), q[2] - 2.0 * c, lo)
        hi, lo = np.where(flat, q[2], hi2), np.where(flat, q[2], lo2)
    return _shift(hi, axis, -1), lo


def _speeds(p, S, G, d, gamma):
    u, _, _, _, bsq = S
    h = p[RHO] + gamma * p[ENY]
    va2, cs2 = bsq / (bsq + h), gamma * (gamma - 1.0) * p[ENY] / h
    cf2 = np.clip(cs2 + va2 - cs2 * va2, 1e-10, 1.0)
    gi = G["gi"]
    A = u[0] ** 2 - (gi[0, 0] + u[0] ** 2) * cf2
    B = 2.0 * (u[d] * u[0] - (gi[0, d] + u[d] * u[0]) * cf2)
    D = u[d] ** 2 - (gi[d, d] + u[d] ** 2) * cf2
    root = np.sqrt(np.maximum(B * B - 4.0 * A * D, 0.0))
    vp, vm = (B - root) / (2.0 * A), (B + root) / (2.0 * A)
    return np.maximum(vp, vm), np.minimum(vp, vm)


def _riemann(p, G, d, cfg, limiter, riemann):
    """Face fluxes and wave speeds along d of one ghosted block."""
    gamma = cfg["gamma"]
    pl, pr = _faces(p, 4 - d, limiter)
    with np.errstate(all="ignore"):
        sl, sr = _state(pl, G), _state(pr, G)
        vl, vr = _speeds(pl, sl, G, d, gamma), _speeds(pr, sr, G, d, gamma)
        cp = np.maximum(np.maximum(0.0, vl[0]), vr[0])
        cm = np.maximum(np.maximum(0.0, -vl[1]), -vr[1])
        cc = np.maximum(cp, cm)
        ul, ur = _flux(pl, sl, G["sg"], 0, gamma), _flux(pr, sr, G["sg"], 0, gamma)
        fl, fr = _flux(pl, sl, G["sg"], d, gamma), _flux(pr, sr, G["sg"], d, gamma)
        if riemann == "laxf":
            f = 0.5 * (fl + fr - cc * (ur - ul))
        else:
            f = (cp * fl + cm * fr - cp * cm * (ur - ul)) / (cp + cm + 1e-20)
        return np.where(G["ok"], f, 0.0), np.where(G["ok"], cc, 0.0)


def _exact_fluxes(case, p, geo, cfg):
    lim, rs = case["limiter"], case["riemann"]
    dim = 3 if case["nx3"] > 1 else 2
    flux = [np.zeros_like(p) for _ in range(dim)]
    alf = np.zeros((p.shape[0], 3, *p.shape[2:]))
    n = p.shape[2:]
    for b, blk in enumerate(_blocks(case)):
        for d in range(1, dim + 1):
            x1 = _axis(cfg, 0, blk[2][0], n[2] - 2 * NG, d == 1)[:n[2]]
            x2 = _axis(cfg, 1, blk[1][0], n[1] - 2 * NG, d == 2)[:n[1]]
            G = geo[b] if d == 3 else _geometry(case["metric"], x1, x2, cfg)
            f, c = _riemann(p[b], G, d, cfg, lim, rs)
            side = 0 if (d == 3 and rs == "hll") else 1
            keep = np.zeros(n, dtype=bool)
            keep[tuple((slice(NG, m - NG + 1) if 3 - ax == d else slice(NG - side, m - NG + side)) if m > 1 else
                       slice(None) for ax, m in enumerate(n))] = True
            flux[d - 1][b] = np.where(keep, f, 0.0)
            alf[b, d - 1] = np.where(keep, c, 0.0)
    return [f.reshape(-1) for f in flux] + [alf.reshape(-1)]


def _exact_ot(case, seed, cycles):
    """RK2 cycles of the Orszag-Tang configuration (MC, LAXF, CT, 1Dvsq with
    the entropy) on one periodic block."""
    cfg = _configs(case, seed)
    P = [_ot_state(case, seed)[0]] * 2
    U = [np.zeros_like(P[0]), np.zeros_like(P[0])]
    n = P[0].shape[1:]
    G = _centre_geometry(case, cfg, next(_blocks(case)))
    inn = (slice(None), *_interior(n))
    gamma = cfg["gamma"]
    dx = [1.0 / case["nx1"], 1.0 / case["nx2"]]
    dt, time = cfg["dt_init"], 0.0
    for _ in range(cycles):
        for c0, c1, beta in ((0, 1, 0.5), (1, 0, 1.0)):
            P[c0] = _fixed(P[c0], G, cfg)[0]
            U[c0] = U[c0].copy()
            U[c0][inn] = _flux(P[c0], _state(P[c0], G), G["sg"], 0, gamma)[inn]
            (f1, a1), (f2, a2) = (_riemann(P[c0], G, d, cfg, "mc", "laxf") for d in (1, 2))
            e = 0.25 * ((f1[BX2] + _shift(f1[BX2], 1, -1)) - (f2[BX1] + _shift(f2[BX1], 2, -1)))
            f1[BX1], f2[BX2] = 0.0, 0.0
            f1[BX2] = 0.5 * (e + _shift(e, 1, 1))
            f2[BX1] = -0.5 * (e + _shift(e, 2, 1))
            div = (_shift(f1, 3, 1) - f1) / dx[0] + (_shift(f2, 2, 1) - f2) / dx[1]
            new = U[c1].copy()
            new[inn] = (U[0] - beta * dt * div)[inn]
            U[c1] = new
            stale = P[c1]
            P[c1] = np.pad(stale[inn], [(0, 0), (0, 0), (NG, NG), (NG, NG)], mode="wrap")
            P[c1][inn] = _isentropic(new[inn], stale[inn], gamma)
        est = 1.0 / sum(1.0 / (cfg["cfl"] * dx[d] / a[inn[1:]].max()) for d, a in enumerate((a1, a2)))
        time, dt = time + dt, min(cfg["dt_factor"] * dt, est)
    return P, U, dt, time


def _isentropic(U, p, gamma):
    """1Dvsq recovery in flat space: v^2 from the entropy K = p[ENT]."""
    D, K = U[RHO], p[8]
    Q0 = U[ENY] - U[RHO]
    Q, B = U[UX1:UX1 + 3], U[BX1:BX1 + 3]
    bsq, qb, qt = (B * B).sum(0), (Q * B).sum(0), (Q * Q).sum(0)
    qt = (-Q0 * Q0 + qt) + Q0 * Q0
    ut = (p[UX1:UX1 + 3] ** 2).sum(0)
    x = 1.0 - 1.0 / (1.0 + ut)

    def w(x):
        rho = D * np.sqrt(1.0 - x)
        pr = K * rho ** gamma
        return rho, pr, (rho + pr / (gamma - 1.0) + pr) / (1.0 - x)

    for _ in range(40):
        rho, pr, W = w(x)
        dW = (gamma * (2.0 - gamma) * pr + (gamma - 1.0) * rho) / (2.0 * (gamma - 1.0) * (1.0 - x) ** 2)
        f = bsq + W
        res = qt - x * f * f + qb * qb * (bsq + 2.0 * W) / (W * W)
        x = np.clip(x + res / (f * (f + 2.0 * dW * (x + qb * qb / W ** 3))), 0.0, 1.0 - 1e-15)
    rho, pr, W = w(x)
    out = p.copy()
    out[RHO], out[ENY] = rho, pr / (gamma - 1.0)
    lor = 1.0 / np.sqrt(1.0 - x)
    for a in range(3):
        out[UX1 + a] = lor / (W + bsq) * (Q[a] + qb * B[a] / W)
        out[BX1 + a] = B[a]
    return out


def exact(case, seed):
    """The result in plain FP64 numpy: the layers, and the Orszag-Tang runs on
    one block.  The torus runs (Christoffel symbols, boundaries and several
    blocks on top of this) are left out."""
    cfg = _configs(case, seed)
    if case["kind"] == "layer":
        p, geo = _layer_state(case, seed)
        n = p.shape[2:]
        if case["layer"] == "fluxes":
            return _exact_fluxes(case, p, geo, cfg)
        if case["layer"] == "fix_cons":
            q, mask = map(np.stack, zip(*(_fixed(p[b], G, cfg) for b, G in enumerate(geo))))
            return [q.reshape(-1), _conserved(q, geo, cfg["gamma"]).reshape(-1), mask.reshape(-1)]
        # the recovered primitives are the ones the conserved state was made of
        out, inn = _guess(p, seed), (slice(None), slice(None), *_interior(n))
        # (no dissipation: K_e only meets its limits)
        out[inn] = p[inn]
        total = p[:, ENT]
        rpow = p[:, RHO] ** (cfg["gamma"] - cfg["gamma_e"])
        g, ge, gp = cfg["gamma"] - 1.0, cfg["gamma_e"] - 1.0, cfg["gamma_p"] - 1.0
        hi = total * rpow / (cfg["ratio_min"] * g / gp + g / ge)
        lo = total * rpow / (cfg["ratio_max"] * g / gp + g / ge)
        kel = np.maximum(lo, np.minimum(p[:, KEL], hi))
        out[:, KEL][inn[1:]] = kel[inn[1:]]
        return [out.reshape(-1), np.zeros(p[:, 0].size, dtype=np.int32)]
    if case.get("problem") != "ot" or case.get("nb1", 1) * case.get("nb2", 1) > 1:
        return None
    cycles = case.get("cycles", 1)
    if case["nx1"] * case["nx2"] * cycles > 400000:
        return None  # more than about 20 seconds of numpy
    P, U, dt, time = _exact_ot(case, seed, cycles)
    if case["kind"] == "step":
        return [P[0][None], dt]
    return [P[0].reshape(-1), U[0].reshape(-1), P[1].reshape(-1), U[1].reshape(-1), np.array([dt, time])]
