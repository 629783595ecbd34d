"""What a user of this framework has it do, as cases that can be timed and checked.

Every case goes through the public entry points (the device classes of op-pic_amd/oppx.py, the serving arena of
op-pic_amd/serve.py, the C-ABI of include/oppx.h) on the sizes of this repository's configurations, tests and
benchmark or between them. FEM-PIC, ensemble, serving and CabanaPIC cases are short segments of a simulation: one
pass starts from the same initial state (a device copy of it), makes a few steps and hands the state back, so that
every pass does the same work. A NESO pass is one step of a periodic population, which does not change in kind. A
field pass is one round of the loops either side of the field solve.

`exact` restates each path in plain torch, in 64 bits, without the framework's code; only the mesh arrays that both
sides get as their input come from the framework's host builders.
"""

import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "op-pic_amd"))

import oppx  # noqa: E402
import serve  # noqa: E402

CHARGE, MASS = 1e-3, 1.0
BOX = ((0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
GONE = oppx.MAX_CELL_INDEX
F64, I32 = torch.float64, torch.int32


def listed():
    return [
        # the smallest simulation (the smoke test's): launches and latency are all there is
        dict(name="fempic_tiny", kind="fempic", loop="fused", nx=4, particles=4_000, steps=10, mesh="x", overlay=2.0,
             cell_order=True, sigma=0.02),
        # the CPU-sized configuration: 48 k tets, 1 M particles in the order they were made, hole fill after each step
        dict(name="fempic_1m", kind="fempic", loop="fused", nx=20, particles=1_000_000, steps=8, mesh="x", overlay=2.0,
             cell_order=False, sigma=0.01),
        # the large single instance at half the benchmark's size: Morton-numbered mesh, particles in cell order, a
        # lazy sort by cell every second step with staged records, hole fill in between
        dict(name="fempic_24m", kind="fempic", loop="periodic", nx=80, particles=24_000_000, steps=6, mesh="morton",
             overlay=1.28, cell_order=True, sigma=0.01),
        # the reference's loop order (push, move, hole fill, deposit: what its generated applications call), no overlay
        dict(name="fempic_loops", kind="fempic", loop="loops", nx=32, particles=1_500_001, steps=4, mesh="x",
             overlay=0.0, cell_order=True, sigma=0.01),
        # one request alone: Sort_All after each step, then the compensated FP32 deposit
        dict(name="fempic_request", kind="fempic", loop="sorted", nx=40, particles=3_000_000, steps=4, mesh="x",
             overlay=2.0, cell_order=True, sigma=0.01),
        # a batched ensemble of independent instances, FP32 deposit, lazy sorts
        dict(name="ensemble_24", kind="ensemble", instances=24, tets_lo=2_000, tets_hi=60_000, parts_lo=10_000,
             parts_hi=400_000, spec=4, steps=4, deposit="f32"),
        # a small ensemble of small instances, FP64 deposit
        dict(name="ensemble_small", kind="ensemble", instances=6, tets_lo=300, tets_hi=3_000, parts_lo=1_000,
             parts_hi=20_000, spec=5, steps=4, deposit="f64"),
        # serving: requests admitted into the arena, stepped together, their results handed back to the host
        dict(name="serving", kind="serving", instances=5, tets_lo=2_000, tets_hi=60_000, parts_lo=20_000,
             parts_hi=300_000, spec=6, steps=6),
        # NESO advection on its periodic grid at half the benchmark's particle count
        dict(name="neso_32m", kind="neso", nx=1024, ny=1024, particles=32_000_000, grid=True, speed=4.0),
        # NESO advection on a mesh that is not taken for the grid: every record is gathered
        dict(name="neso_gathered", kind="neso", nx=300, ny=220, particles=1_500_000, grid=False, speed=4.0),
        # CabanaPIC's two-stream deck, a smaller box at the deck's 750 particles a cell
        dict(name="cabana_9m", kind="cabana", nx=20, ny=20, nz=30, per_cell=750, steps=4),
        # the loops either side of the field solve, on the mesh of a mid-sized instance
        dict(name="field_1m", kind="field", nx=60),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fempic", "fempic", "fempic", "ensemble", "serving", "neso", "cabana", "field"])
    if kind == "fempic":
        return dict(kind=kind, loop=rng.choice(["fused", "periodic", "loops", "sorted"]), nx=rng.randint(3, 48),
                    particles=_spread(rng, 1_000, 6_000_000), steps=rng.randint(2, 8), mesh=rng.choice(["x", "morton"]),
                    overlay=rng.choice([0.0, 1.0, 1.28, 2.0]), cell_order=rng.random() < 0.7,
                    sigma=rng.choice([0.005, 0.01, 0.02]))
    if kind in ("ensemble", "serving"):
        lo, parts = _spread(rng, 100, 10_000), _spread(rng, 1_000, 40_000)
        case = dict(kind=kind, instances=rng.randint(2, 24 if kind == "ensemble" else 6), tets_lo=lo,
                    tets_hi=lo * rng.randint(2, 6), parts_lo=parts, parts_hi=parts * rng.randint(2, 8),
                    spec=rng.randint(1, 1 << 20), steps=rng.randint(2, 6))
        return dict(case, deposit=rng.choice(["f32", "f64"])) if kind == "ensemble" else case
    if kind == "neso":
        return dict(kind=kind, nx=_spread(rng, 8, 1024), ny=_spread(rng, 8, 1024),
                    particles=_spread(rng, 2_000, 16_000_000), grid=rng.random() < 0.6, speed=rng.choice([0.5, 4.0]))
    if kind == "cabana":
        return dict(kind=kind, nx=rng.randint(2, 24), ny=rng.randint(2, 24), nz=rng.randint(2, 24),
                    per_cell=rng.choice([2, 40, 150, 750]), steps=rng.randint(1, 4))
    return dict(kind=kind, nx=rng.randint(4, 60))


# ---- inputs ---------------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=6)
def _mesh(nx, order, overlay):
    """Box mesh, field and (overlay > 0) direct-hop overlay of 1 / round(overlay * nx) spacing: no seed in them."""
    m = oppx.box_mesh(nx, nx, nx, order=order)
    gs = 1.0 / max(1, int(round(overlay * nx))) if overlay > 0 else None
    return m, oppx.box_field_sines(m), None if gs is None else oppx.dh_overlay(m, *BOX, gs), gs


def _instance(nx, particles, seed, sigma, order="x", overlay=2.0, cell_order=True):
    m, ef, ov, gs = _mesh(nx, order, overlay)
    pos, vel, p2c = oppx.box_particles(particles, seed, sigma, m)
    if cell_order:
        at = torch.argsort(torch.from_numpy(p2c).to(_dev()), stable=True).cpu().numpy()
        pos, vel, p2c = pos[at], vel[at], p2c[at]
    d = dict(mesh=m, ef=ef, pos=pos, vel=vel, p2c=p2c, charge=CHARGE, mass=MASS,
             dt=0.5 / nx / (sigma * math.sqrt(3.0)))
    return dict(d, overlay=ov, bmin=BOX[0], bmax=BOX[1], gs=gs) if ov is not None else d


def _fempic_instance(c, seed):
    return _instance(c["nx"], c["particles"], seed, c["sigma"], c["mesh"], c["overlay"], c["cell_order"])


def _specs(c):
    """(nx, particles, sigma) of an ensemble's or a stream's instances; the case's `spec` fixes them."""
    r = np.random.default_rng(c["spec"])
    log = lambda lo, hi: math.exp(r.uniform(math.log(lo), math.log(hi)))
    return [(max(2, int(round((log(c["tets_lo"], c["tets_hi"]) / 6.0) ** (1.0 / 3.0)))),
             int(log(c["parts_lo"], c["parts_hi"])), float(r.uniform(0.005, 0.02))) for _ in range(c["instances"])]


def _instances(c, seed):
    return [_instance(nx, n, seed * 1009 + i, sigma) for i, (nx, n, sigma) in enumerate(_specs(c))]


def _neso_inputs(c, seed):
    cw, dt = 0.5, 0.5
    m = oppx.neso_mesh(c["nx"], c["ny"], cw)
    return (m, dt) + oppx.neso_particles(c["particles"], seed, m, c["speed"] * cw / dt)


def _cabana_inputs(c, seed):
    """The two-stream deck (bench.py) with a little seeded velocity spread and seeded synthetic fields."""
    nx, ny, nz, nppc = c["nx"], c["ny"], c["nz"], c["per_cell"]
    v0, nc = 0.0866025403784439, nx * ny * nz
    gam = 1.0 / math.sqrt(1.0 - v0 * v0)
    dims = [1.0 / nx, 0.628318530717959 * gam * math.sqrt(gam) / ny, 1.0 / nz]
    dt = 0.99 / math.sqrt(sum(d ** -2 for d in dims))
    g = torch.Generator(device=_dev()).manual_seed(seed)
    k = torch.arange(nc * nppc, device=_dev())
    cell = k // nppc
    pos = torch.zeros((3, nc * nppc), dtype=F64, device=_dev())
    pos[1] = ((2 * (k // 2)) % nppc).to(F64) * (2.0 / nppc) + 1.0 / nppc - 1.0
    vel = 1e-3 * torch.randn((3, nc * nppc), dtype=F64, device=_dev(), generator=g)
    vel[0] += torch.where(k % 2 == 0, 1.0, -1.0).to(F64) * v0 * gam
    i = np.arange(nc)
    ix, iy, iz = i % nx, (i // nx) % ny, i // (nx * ny)
    at = lambda a, b, e: (a % nx) + nx * ((b % ny) + ny * (e % nz))
    c2c6 = np.stack([at(ix - 1, iy, iz), at(ix, iy - 1, iz), at(ix, iy, iz - 1), at(ix + 1, iy, iz), at(ix, iy + 1, iz),
                     at(ix, iy, iz + 1)], axis=1).astype(np.int32)
    scale = torch.tensor([0.5, 0.2, 0.2, 0.1] * 3 + [0.5, 0.2] * 3, dtype=F64, device=_dev())
    interp = torch.randn((nc, 18), dtype=F64, device=_dev(), generator=g) * scale
    weight = torch.full((nc * nppc,), 2.0 * dims[0] * dims[1] * dims[2] / nppc, dtype=F64, device=_dev())
    return dict(pos=pos, vel=vel, weight=weight, p2c=cell.to(I32), c2c6=torch.from_numpy(c2c6).to(_dev()), interp=interp,
                qsp=-1.0, qdt_2mc=-dt / 2.0, cdt_d=[dt / d for d in dims], n_cells=nc)


def _field_inputs(c, seed):
    m = _mesh(c["nx"], "x", 0.0)[0]
    nn, nc = m["n_nodes"], m["n_cells"]
    g = torch.Generator(device=_dev()).manual_seed(seed)
    new = lambda *shape: torch.randn(shape, dtype=F64, device=_dev(), generator=g)
    return dict(m=m, nn=nn, nc=nc, c2n=torch.from_numpy(m["c2n"]).to(_dev()), ef=new(nc, 3), sd=new(nc, 12), pot=new(nn),
                rho=new(nn).abs(), vol=new(nn).abs() + 0.1,
                kind=torch.randint(0, 4, (nn,), dtype=I32, device=_dev(), generator=g))


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


# ---- prepare and run ------------------------------------------------------------------------------------------

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "fempic":
        d = _fempic_instance(c, seed)
        more = {k: d[k] for k in ("overlay", "bmin", "bmax", "gs") if k in d}
        return dict(c=c, dt=d["dt"], proto=oppx.FempicDevice(d["mesh"], d["ef"], d["pos"], d["vel"], d["p2c"], **more))
    if kind == "ensemble":
        return dict(c=c, proto=oppx.FempicBatch(_instances(c, seed)))
    if kind == "serving":
        tpl = [serve.Template.of(d).make_resident() for d in _instances(c, seed)]
        total = lambda key: sum(getattr(t, key) for t in tpl)
        # room for a second stream's particles beside the first one's, which leave the set at the next sort
        arena = serve.FempicArena(total("n_cells"), total("n_nodes"), 2 * total("n_part"), total("overlay_words"), 64)
        return dict(c=c, templates=tpl, arena=arena)
    if kind == "neso":
        m, dt, pos, vel, p2c = _neso_inputs(c, seed)
        return dict(c=c, dt=dt, dev=oppx.NesoDevice(m, pos, vel, p2c, grid=c["grid"]))
    if kind == "cabana":
        d = _cabana_inputs(c, seed)
        n = d["p2c"].numel()
        d.update(now=[d[k].clone() for k in ("pos", "vel", "p2c")], streak=torch.zeros_like(d["pos"]),
                 acc=torch.zeros((d["n_cells"], 12), dtype=F64, device=_dev()),
                 counters=torch.zeros(oppx.COUNTER_WORDS, dtype=I32, device=_dev()))
        d["counters"][0] = n
        pos, vel, p2c = d["now"]
        d["parts"] = oppx.CabanaParts(n, pos.data_ptr(), vel.data_ptr(), d["streak"].data_ptr(), d["weight"].data_ptr(),
                                      p2c.data_ptr())
        d["mesh"] = oppx.CabanaMesh(d["n_cells"], d["c2c6"].data_ptr(), d["interp"].data_ptr())
        return dict(c=c, d=d)
    d = _field_inputs(c, seed)
    d["out"] = dict(ef=d["ef"].clone(), rho=d["rho"].clone(), bnd=torch.zeros_like(d["pot"]),
                    top=torch.zeros(2, dtype=F64, device=_dev()))
    d["bytes"] = int(oppx.lib().oppx_max_scratch_bytes(3 * d["nc"]))
    d["scratch"] = torch.zeros(d["bytes"], dtype=torch.uint8, device=_dev())
    return dict(c=c, d=d)


def run(state):
    return _RUN[state["c"]["kind"]](state)


def _run_fempic(s):
    c, g = s["c"], s["proto"].clone()
    for k in range(c["steps"]):
        if c["loop"] == "fused":
            g.step_fused(CHARGE, MASS, s["dt"])
        elif c["loop"] == "loops":
            g.step_unfused(CHARGE, MASS, s["dt"], record_hops=False)
        elif c["loop"] == "periodic":
            sort = k % 2 == 1
            g.step_begin()
            g.pass_fused(CHARGE, MASS, s["dt"], stage=sort)
            g.sort(drop_removed=True, lazy=True) if sort else g.holefill()
        else:
            g.step_begin()
            g.pass_fused(CHARGE, MASS, s["dt"], deposit=False)
            g.sort(drop_removed=True)
            g.deposit_sorted_f32()
    g.materialize()
    return _state(g, g.sync_size(), g.charge_f32 if c["loop"] == "sorted" else g.charge)


def _state(g, n, charge):
    """The particle dats, their slots past the n live ones cleared (what they hold is not defined), and the charge."""
    for t in (g.pos, g.vel, g.lc):
        t[:, n:].zero_()
    g.p2c[n:].fill_(GONE)
    return dict(pos=g.pos, vel=g.vel, lc=g.lc, p2c=g.p2c, charge=charge)


def _run_ensemble(s):
    c, g = s["c"], s["proto"].clone()
    g.steps_batch(c["steps"], c["deposit"])
    return _state(g, g.sync_size(), g.charge_f32 if c["deposit"] == "f32" else g.charge)


def _run_serving(s):
    c, arena = s["c"], s["arena"]
    slots = [arena.admit(t) for t in s["templates"]]
    for _ in range(c["steps"]):
        arena.step()
    got = arena.retire(slots)  # every request's results, on the host
    # their lengths differ from seed to seed; what they were copied from is the arena's state, which retire leaves
    return dict(_state(arena, arena.size, arena.charge_f32), counts=[r["n"] for r in got])


def _run_neso(s):
    g = s["dev"]
    g.step(s["dt"])
    return dict(pos=g.pos, mdir=g.mdir, p2c=g.p2c)


def _run_cabana(s):
    d = s["d"]
    for to, key in zip(d["now"], ("pos", "vel", "p2c")):
        to.copy_(d[key])
    cdt = (ctypes.c_double * 3)(*d["cdt_d"])
    for _ in range(s["c"]["steps"]):
        d["acc"].zero_()
        oppx.check(oppx.lib().oppx_cabana_move_deposit(
            d["p2c"].numel(), ctypes.byref(d["parts"]), ctypes.byref(d["mesh"]), d["acc"].data_ptr(), d["qsp"],
            d["qdt_2mc"], cdt, d["counters"].data_ptr(), None, torch.cuda.current_stream().cuda_stream), "cabana")
    return dict(pos=d["now"][0], vel=d["now"][1], p2c=d["now"][2], acc=d["acc"])


def _run_field(s):
    d = s["d"]
    L, o, stream = oppx.lib(), d["out"], torch.cuda.current_stream().cuda_stream
    nc, nn = d["nc"], d["nn"]
    o["ef"].copy_(d["ef"])
    o["rho"].copy_(d["rho"])
    oppx.check(L.oppx_fempic_boundary_potential(nn, d["kind"].data_ptr(), -0.75, o["bnd"].data_ptr(), stream), "bnd")
    oppx.check(L.oppx_fempic_node_charge_density(nn, o["rho"].data_ptr(), d["vol"].data_ptr(), 2.5, stream), "rho")
    oppx.check(L.oppx_fempic_electric_field(nc, o["ef"].data_ptr(), d["sd"].data_ptr(), d["c2n"].data_ptr(),
                                            d["pot"].data_ptr(), nn, None, stream), "ef")
    for k, (n, x, signed) in enumerate(((3 * nc, o["ef"], 1), (nn, d["pot"], 0))):
        oppx.check(L.oppx_max_reduce(n, x.data_ptr(), signed, 0.0, o["top"][k:].data_ptr(), d["scratch"].data_ptr(),
                                     d["bytes"], stream), "max")
    return dict(o)


_RUN = dict(fempic=_run_fempic, ensemble=_run_ensemble, serving=_run_serving, neso=_run_neso, cabana=_run_cabana,
            field=_run_field)


# ---- what a pass cannot do without ----------------------------------------------------------------------------

def work(case):
    """Each input read once and each output written once, a step: per FEM-PIC particle pos, vel, p2c in and out and lc
    out, 192 B a tet and 16 B a node (the benchmark's count), 36 B a particle more for a deposit of its own."""
    c, kind = case, case["kind"]
    if kind in ("fempic", "ensemble", "serving"):
        sizes = [(c["nx"], c["particles"])] if kind == "fempic" else [(nx, n) for nx, n, _ in _specs(c)]
        n, nc, nn = sum(p for _, p in sizes), sum(6 * x ** 3 for x, _ in sizes), sum((x + 1) ** 3 for x, _ in sizes)
        own = kind == "serving" or c.get("deposit") == "f32" or c.get("loop") in ("loops", "sorted")
        bytes_ = c["steps"] * ((172 if own else 136) * n + 192 * nc + 16 * nn)
        if kind == "serving":
            bytes_ += 84 * n
        return dict(bytes=bytes_, flops=c["steps"] * 110 * n)
    if kind == "neso":
        return dict(bytes=64 * c["particles"] + 32 * c["nx"] * c["ny"], flops=40 * c["particles"])
    if kind == "cabana":
        nc = c["nx"] * c["ny"] * c["nz"]
        return dict(bytes=c["steps"] * (160 * nc * c["per_cell"] + 360 * nc), flops=c["steps"] * 250 * nc * c["per_cell"])
    nc, nn = 6 * c["nx"] ** 3, (c["nx"] + 1) ** 3
    return dict(bytes=(24 + 96 + 16 + 24) * nc + (8 + 24 + 12 + 8) * nn, flops=24 * nc + 2 * nn)


# ---- the same in plain torch, in 64 bits ----------------------------------------------------------------------

def _t(a, dtype=F64):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev(), dtype=dtype)


class _Box:
    """One FEM-PIC instance in plain torch: push, direct hop, walk, removal and the finalize, step by step."""

    def __init__(self, d):
        m = d["mesh"]
        self.det, self.c2 = _t(m["c_det"]).reshape(-1, 16), (1.0 / 6.0) / _t(m["c_vol"])
        self.c2c, self.c2n = _t(m["c2c"], torch.int64), _t(m["c2n"], torch.int64)
        self.ef, self.nn, self.dt = _t(d["ef"]), m["n_nodes"], d["dt"]
        self.pos, self.vel, self.cell = _t(d["pos"]), _t(d["vel"]), _t(d["p2c"], torch.int64)
        self.lc = torch.zeros((len(d["p2c"]), 4), dtype=F64, device=_dev())
        self.overlay = None
        if "overlay" in d:
            self.overlay, self.gs = _t(d["overlay"], torch.int64), d["gs"]
            self.dims = [int(v) for v in oppx.dh_dims(d["bmin"], d["bmax"], d["gs"])]

    def weights(self, p, cell):
        a = self.det[cell].reshape(-1, 4, 4)
        return self.c2[cell][:, None] * (a[:, :, 0] - a[:, :, 1] * p[:, :1] + a[:, :, 2] * p[:, 1:2] - a[:, :, 3] * p[:, 2:])

    def step(self, fill):
        self.vel = self.vel + (CHARGE / MASS * self.dt) * self.ef[self.cell]
        self.pos = self.pos + self.vel * self.dt
        cell = self.cell
        if self.overlay is not None:
            t = self.pos * (1.0 / self.gs)
            top = torch.tensor(self.dims, dtype=F64, device=_dev())
            inside = ((t > -1.0) & (t < top)).all(1)
            i = t.trunc().clamp(min=0).minimum(top - 1).to(torch.int64)
            cell = self.overlay[i[:, 0] + self.dims[0] * (i[:, 1] + self.dims[1] * i[:, 2])]
            cell = torch.where(inside, cell, GONE)
        on = (cell != GONE).nonzero()[:, 0]
        while on.numel():
            still = []
            for part in on.split(1 << 22):
                l = self.weights(self.pos[part], cell[part])
                self.lc[part] = l
                out = ~((l > -1e-10) & (l - 1.0 < 1e-10)).all(1)
                part, l = part[out], l[out]
                nb = self.c2c[cell[part]].gather(1, l.argmin(1)[:, None])[:, 0]
                cell[part] = torch.where(nb < 0, GONE, nb)
                still.append(part[nb >= 0])
            on = torch.cat(still)
        gone = cell == GONE
        n = cell.numel()
        if fill == "sort":
            keep = torch.argsort(cell, stable=True)[:n - int(gone.sum())]
        else:  # the k-th hole below the new size takes the k-th live particle from the end
            size = n - int(gone.sum())
            keep = torch.arange(size, device=_dev())
            holes = gone[:size].nonzero()[:, 0]
            keep[holes] = ((~gone[size:]).nonzero()[:, 0] + size).flip(0)
        self.pos, self.vel, self.lc, self.cell = self.pos[keep], self.vel[keep], self.lc[keep], cell[keep]

    def charge(self):
        q = torch.zeros(self.nn, dtype=F64, device=_dev())
        return q.index_add_(0, self.c2n[self.cell].reshape(-1), self.lc.reshape(-1))

    def out(self):
        return dict(pos=self.pos.T, vel=self.vel.T, lc=self.lc.T, p2c=None, charge=self.charge())


def _padded(out, slots):
    """A state in `slots` particle slots, the ones past the live particles cleared as _state() clears them."""
    pad = lambda t: torch.nn.functional.pad(t, (0, slots - t.shape[1]))
    return dict(out, **{k: pad(out[k]) for k in ("pos", "vel", "lc")})


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _exact_fempic(c, seed):
    b = _Box(_fempic_instance(c, seed))
    for k in range(c["steps"]):
        b.step("sort" if c["loop"] == "sorted" or (c["loop"] == "periodic" and k % 2 == 1) else "hole")
    return _padded(b.out(), c["particles"])


def _exact_instances(c, seed):
    boxes = []
    for d in _instances(c, seed):
        b = _Box(d)
        for _ in range(c["steps"]):
            b.step("sort")
        boxes.append(b.out())
    cat = {k: torch.cat([b[k] for b in boxes], dim=-1) for k in ("pos", "vel", "lc", "charge")}
    slots = sum(n for _, n, _ in _specs(c))
    return dict(_padded(cat, 2 * slots if c["kind"] == "serving" else slots), p2c=None)


def _exact_neso(c, seed):
    m, dt, pos, vel, _ = _neso_inputs(c, seed)
    ext = torch.tensor([c["nx"] * m["cell_width"], c["ny"] * m["cell_width"]], dtype=F64, device=_dev())[:, None]
    p = _t(pos.T) + _t(vel.T) * dt
    t = p + (p.abs() + 2.0).trunc() * ext
    return dict(pos=t - ext * (t / ext).trunc(), mdir=None, p2c=None)


def _exact_cabana(c, seed):
    d = _cabana_inputs(c, seed)
    p, v, cell = d["pos"].T.contiguous(), d["vel"].T.contiguous(), d["p2c"].to(torch.int64)
    cdt, c2c6 = torch.tensor(d["cdt_d"], dtype=F64, device=_dev()), d["c2c6"].to(torch.int64)
    q = d["weight"] * d["qsp"]
    acc = None
    for _ in range(c["steps"]):
        acc = torch.zeros((d["n_cells"] * 12,), dtype=F64, device=_dev())
        f = d["interp"][cell]
        x, y, z = p[:, 0], p[:, 1], p[:, 2]
        e = torch.stack([f[:, 0] + y * f[:, 1] + z * (f[:, 2] + y * f[:, 3]), f[:, 4] + z * f[:, 5] + x * (f[:, 6] + z * f[:, 7]),
                         f[:, 8] + x * f[:, 9] + y * (f[:, 10] + x * f[:, 11])], 1)
        b = torch.stack([f[:, 12] + x * f[:, 13], f[:, 14] + y * f[:, 15], f[:, 16] + z * f[:, 17]], 1)
        h = d["qdt_2mc"] * e
        u = v + h
        t = d["qdt_2mc"] / torch.sqrt(1.0 + (u * u).sum(1))
        bb = (b * b).sum(1)
        w = t * t * bb
        r3 = t * (1.0 + w * (1.0 / 3.0 + w * 2.0 / 15.0))
        r4 = 2.0 * r3 / (1.0 + bb * r3 * r3)
        u = u + r4[:, None] * torch.linalg.cross(u + r3[:, None] * torch.linalg.cross(u, b), b)
        v = u + h
        left = 2.0 * v * cdt / torch.sqrt(1.0 + (v * v).sum(1))[:, None]  # the whole track, in cell units
        on = torch.arange(cell.numel(), device=_dev())
        while on.numel():  # one streak a round: to the first face on the way, or to the track's end
            s, a = left[on], p[on]
            way = torch.where(s > 0, 1.0, -1.0).to(F64)
            frac, axis = torch.where(s == 0, math.inf, (way - a) / s).min(1)
            end = frac >= 1.0
            half = 0.5 * s * frac.clamp(max=1.0)[:, None]
            mid = a + half
            w = q[on] * half.prod(1) / 3.0
            for k in range(3):
                i, j = (k + 1) % 3, (k + 2) % 3
                g = q[on] * half[:, k]
                terms = [g * (1 - mid[:, i]) * (1 - mid[:, j]) + w, g * (1 + mid[:, i]) * (1 - mid[:, j]) - w,
                         g * (1 - mid[:, i]) * (1 + mid[:, j]) - w, g * (1 + mid[:, i]) * (1 + mid[:, j]) + w]
                for n, value in enumerate(terms):
                    acc.index_add_(0, cell[on] * 12 + 4 * k + n, value)
            p[on], left[on] = a + 2.0 * half, s - 2.0 * half
            on, axis, way = on[~end], axis[~end], way[~end]
            d_axis = way.gather(1, axis[:, None])[:, 0]
            p[on, axis] = -d_axis
            cell[on] = c2c6[cell[on], axis + torch.where(d_axis > 0, 3, 0)]
    return dict(pos=p.T, vel=v.T, p2c=None, acc=acc.reshape(-1, 12))


def _exact_field(c, seed):
    d = _field_inputs(c, seed)
    phi = d["pot"][d["c2n"].to(torch.int64)]
    ef = d["ef"] - (d["sd"].reshape(-1, 4, 3) * phi[:, :, None]).sum(1)
    bnd = torch.where(d["kind"] == 3, 0.75, 0.0).to(F64)
    top = torch.stack([ef.abs().max(), d["pot"].max().clamp(min=0.0)])
    return dict(ef=ef, rho=d["rho"] * (2.5 / d["vol"]), bnd=bnd, top=top)


_EXACT = dict(fempic=_exact_fempic, ensemble=_exact_instances, serving=_exact_instances, neso=_exact_neso,
              cabana=_exact_cabana, field=_exact_field)
