"""Workloads of the particle path, of the field operators beside it and of
whole cycles, as a program that uses this package runs them.

A case names an operation (``op``), a precision, a grid, particles per cell
and what the operation leaves open:

``caller``   the reference's own call sequence on particles in the caller's
             arrays: mover_PC, setZeroSpeciesDensities, interpP2G (or the
             fused mover_interp), optionally particle_sort.
``phase``    one or more phases of the tile-resident Engine, optionally
             after a re-sort (the inner loop of a long run).
``batch``    one phase of several independent instances (Batch).
``handover`` particles that live in the caller's arrays between steps:
             Engine.load, a phase or a deposit, Engine.store.
``cycle``    a whole cycle around the solver: the engine's phase, the ghost
             fold, the sum over species, the net rhoc, the hat densities and
             applications of the Maxwell operator.
``fields``   the field side of that cycle alone.

Particles start as the Harris sheet's lattice (cell by cell, four species or
multiples of them) and have streamed freely for ``age`` steps, as in the
middle of a run; ``order`` says whether they are still in the order of the
initial condition ("load"), were put in bins since ("binned") or come in no
order at all ("random").
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import sputnipic_amd as S

DEV = "cuda"
COMPONENTS = ("x", "y", "z", "u", "v", "w", "q")
DT, C_LIGHT, FOURPI, THETA = 0.25, 1.0, 12.5663706144, 1.0
# qom, density, thermal speed, drift along z, current-sheet profile: the
# four species of the 3-D Harris sheet
SPECIES = (
    (-64.0, 1.0, 0.045, 0.0065, True),
    (1.0, 1.0, 0.0126, -0.0325, True),
    (-64.0, 0.1, 0.045, 0.0, False),
    (1.0, 0.1, 0.0126, 0.0, False),
)
PERIODIC = (True, False, True)
CELL = 20.0 / 128.0  # cell edge of the 128x64x64 sheet on its 20x10x10 box


def _case(name, op, prec, grid, ppc, **more):
    d = {"name": name, "op": op, "prec": prec, "nx": grid[0], "ny": grid[1], "nz": grid[2],
         "ppcx": ppc[0], "ppcy": ppc[1], "ppcz": ppc[2], "species": 4, "cell": CELL, "age": 40,
         "order": "load", "waits": True}
    d.update(more)
    return d


def listed():
    return [
        # the reference's calls at the size of a smoke test: launches, waits
        # and status reads are all there is
        _case("caller_f64_tiny", "caller", "f64", (16, 8, 8), (2, 2, 2), calls="separate"),
        # the reference's calls, species by species, on the particles of an
        # ordinary run between two of its sorts
        _case("caller_mover_f64", "caller", "f64", (96, 48, 48), (3, 3, 3), species=1,
              calls="mover", age=20),
        _case("caller_deposit_f64", "caller", "f64", (96, 48, 48), (3, 3, 3), species=1,
              calls="deposit", order="binned"),
        _case("caller_fused_f32", "caller", "f32", (61, 35, 31), (3, 3, 3), species=1,
              calls="fused", age=8),
        # the binned sort of the reference, after a push as it runs there
        _case("caller_sort_f64", "caller", "f64", (64, 32, 32), (4, 4, 4), species=1,
              calls="sort", order="binned"),
        # a small ragged run through one whole cycle
        _case("cycle_f64_small", "cycle", "f64", (33, 17, 19), (3, 3, 3), images=8, waits=False),
        # field operators on the grid of the sheet
        _case("fields_f64_gem", "fields", "f64", (128, 64, 64), (1, 1, 1), images=8, waits=False),
        # particles handed over to the engine and back on each step
        _case("handover_f64", "handover", "f64", (63, 32, 31), (4, 4, 4), push=True),
        # independent instances of different sizes in one launch
        _case("batch_f32_12", "batch", "f32", (32, 16, 16), (2, 3, 3), instances=12, waits=False),
        # eight species, re-sorted every five phases
        _case("phase_f32_8species", "phase", "f32", (64, 64, 48), (2, 4, 4), species=8, phases=5,
              resort=True, waits=False),
        # the published run, 262 million particles, in both precisions
        _case("phase_f64_gem", "phase", "f64", (128, 64, 64), (5, 5, 5), phases=1, resort=False,
              waits=False),
        _case("phase_f32_gem", "phase", "f32", (128, 64, 64), (5, 5, 5), phases=1, resort=False,
              waits=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grid(rng, lo, hi):
    """A grid of about lo..hi cells, sides of any parity, x the longest."""
    n = _log(rng, lo, hi)
    side = (n / 2.0) ** (1.0 / 3.0)
    y = max(4, int(round(side * rng.uniform(0.8, 1.25))))
    z = max(4, int(round(side * rng.uniform(0.8, 1.25))))
    x = max(4, int(round(n / (y * z))))
    return x, y, z


def draw(rng):
    op = rng.choice(("caller", "caller", "phase", "phase", "batch", "handover", "cycle", "fields"))
    prec = "f64" if op in ("cycle", "fields") else rng.choice(("f64", "f32"))
    more = {"cell": round(CELL * _log(rng, 1.0, 3.0), 6), "age": int(_log(rng, 4, 120)),
            "waits": rng.random() < 0.5}
    ppc = (rng.randint(1, 4), rng.randint(1, 4), rng.randint(1, 4))
    if op == "caller":
        grid = _grid(rng, 1000, 200000)
        while grid[0] * grid[1] * grid[2] * ppc[0] * ppc[1] * ppc[2] > 6e6:
            ppc = (rng.randint(1, 4), rng.randint(1, 4), rng.randint(1, 4))
        more.update(species=1, order=rng.choice(("load", "binned", "random")),
                    calls=rng.choice(("separate", "mover", "deposit", "fused", "sort")))
    elif op == "phase":
        grid = _grid(rng, 1000, 400000)
        ppc = (rng.randint(1, 5), rng.randint(2, 5), rng.randint(2, 5))
        more.update(species=rng.choice((1, 2, 4, 4, 8)), phases=rng.randint(1, 5),
                    resort=rng.random() < 0.3)
        n = grid[0] * grid[1] * grid[2] * ppc[0] * ppc[1] * ppc[2]
        if n * more["species"] * more["phases"] > 2e8:
            more["phases"] = 1
        while n * more["species"] > 2e8:
            more["species"] //= 2
    elif op == "batch":
        grid = _grid(rng, 1000, 16000)
        more.update(instances=rng.randint(2, 16))
    elif op == "handover":
        grid = _grid(rng, 1000, 100000)
        more.update(push=rng.random() < 0.5, order=rng.choice(("load", "binned", "random")))
    else:
        grid = _grid(rng, 2000, 400000)
        more.update(images=rng.randint(1, 16))
        if op == "cycle":
            ppc = (rng.randint(1, 3), rng.randint(1, 3), rng.randint(1, 3))
        else:
            ppc = (1, 1, 1)
    d = _case("", op, prec, grid, ppc, **more)
    del d["name"]
    return d


# ---- inputs -----------------------------------------------------------------


class _Box:
    """Grid constants of a case's box, as any program around it knows them."""

    def __init__(self, nx, ny, nz, cell):
        self.n = (nx, ny, nz)
        self.d = (cell, cell, cell)
        self.L = (nx * cell, ny * cell, nz * cell)
        self.nodes = (nx + 3, ny + 3, nz + 3)
        self.cells = nx * ny * nz


def _box(case, k=0):
    # instance k of a batch: grids of scale 1 to 3 halves, box unchanged
    s = 1.0 + 0.125 * (k % 5)
    n = [max(4, int(round(case[a] * s))) for a in ("nx", "ny", "nz")]
    return _Box(*n, case["cell"])


def _species(case, s):
    return SPECIES[s % len(SPECIES)]


def _count(case, box):
    return box.cells * case["ppcx"] * case["ppcy"] * case["ppcz"]


def _dtype(case):
    return torch.float64 if case["prec"] == "f64" else torch.float32


def _node_axes(box):
    return [(torch.arange(n, device=DEV, dtype=torch.float64) - 1.0) * d
            for n, d in zip(box.nodes, box.d)]


def _field_arrays(case, box, seed):
    """Harris-sheet magnetic field with a perturbation, and the electric
    field of a weak static potential, on the nodes."""
    g = torch.Generator().manual_seed(7919 * seed + 17)
    ph = torch.rand(6, generator=g, dtype=torch.float64).tolist()
    x, y, z = _node_axes(box)
    X, Y, Z = x[:, None, None], y[None, :, None], z[None, None, :]
    Lx, Ly, Lz = box.L
    tau = 2.0 * math.pi
    one = torch.ones(box.nodes, device=DEV, dtype=torch.float64)
    b0 = 0.0195
    amp = b0 * (0.02 + 0.04 * ph[0])
    yc = (Y - 0.5 * Ly) / (0.05 * Ly)
    a1 = tau * (X / Lx + ph[1])
    a2 = tau * (Z / Lz + ph[2])
    f = {
        "Bxn": b0 * torch.tanh(yc) * one + amp * torch.sin(a1) * torch.cos(a2),
        "Byn": amp * torch.sin(a1 + 0.3) * torch.cos(a2) * one,
        "Bzn": 0.1 * b0 * one + amp * torch.cos(a1) * torch.sin(a2),
    }
    phi0 = 1e-5 * (0.5 + ph[3])  # qom phi0 stays below the thermal energy
    b1 = tau * (X / Lx + ph[4])
    b2 = tau * (Z / Lz + ph[5])
    cy = torch.sin(math.pi * Y / Ly)
    f["Ex"] = -phi0 * tau / Lx * torch.cos(b1) * cy * torch.cos(b2)
    f["Ey"] = -phi0 * math.pi / Ly * torch.sin(b1) * torch.cos(math.pi * Y / Ly) * torch.cos(b2)
    f["Ez"] = phi0 * tau / Lz * torch.sin(b1) * cy * torch.sin(b2)
    dt = _dtype(case)
    return {k: v.to(dt).contiguous() for k, v in f.items()}


def _inside(p, L, periodic):
    if periodic:
        return torch.remainder(p, L)
    p = torch.remainder(p, 2.0 * L)
    return torch.where(p > L, 2.0 * L - p, p)


def _particle_arrays(case, box, s, seed):
    """Species s: the lattice of the initial condition, cell by cell,
    thermal velocities, streamed freely for `age` steps."""
    qom, rho, uth, w0, sheet = _species(case, s)
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 101 * s + 1)
    n = _count(case, box)
    px, py, pz = case["ppcx"], case["ppcy"], case["ppcz"]
    idx = torch.arange(n, device=DEV)
    sub = torch.remainder(idx, px * py * pz)
    c = torch.div(idx, px * py * pz, rounding_mode="floor")
    del idx
    axis = {}
    ny, nz = box.n[1], box.n[2]
    axis["z"] = ((torch.remainder(c, nz) + (torch.remainder(sub, pz) + 0.5) / pz) * box.d[2])
    c = torch.div(c, nz, rounding_mode="floor")
    sub = torch.div(sub, pz, rounding_mode="floor")
    axis["y"] = ((torch.remainder(c, ny) + (torch.remainder(sub, py) + 0.5) / py) * box.d[1])
    c = torch.div(c, ny, rounding_mode="floor")
    sub = torch.div(sub, py, rounding_mode="floor")
    axis["x"] = (c + (sub + 0.5) / px) * box.d[0]
    del c, sub
    out = {}
    yr = (axis["y"] - 0.5 * box.L[1]) / (0.05 * box.L[1])
    dens = rho / torch.cosh(yr) ** 2 if sheet else torch.full_like(yr, rho)
    del yr
    sign = 1.0 if qom > 0 else -1.0
    vol = box.d[0] * box.d[1] * box.d[2]
    out["q"] = (sign / FOURPI / (px * py * pz)) * dens * vol
    del dens
    for a, v, k, L in (("x", "u", 0, box.L[0]), ("y", "v", 1, box.L[1]), ("z", "w", 2, box.L[2])):
        vel = torch.randn(n, generator=g, device=DEV, dtype=torch.float64) * uth
        if v == "w":
            vel += w0
        out[v] = vel
        out[a] = _inside(axis.pop(a) + vel * (DT * case["age"]), L, PERIODIC[k])
    dt = _dtype(case)
    out = {k: out[k].to(dt) for k in COMPONENTS}
    if case["order"] == "binned":
        perm = torch.sort(_bins(box, out["x"], out["y"], out["z"]), stable=True).indices
        out = {k: v[perm] for k, v in out.items()}
    elif case["order"] == "random":
        perm = torch.randperm(n, generator=g, device=DEV)
        out = {k: v[perm] for k, v in out.items()}
    return out


SORT_CPS = 4


def _bins(box, x, y, z):
    """Bin of particle_sort: sort_cps guard-inclusive cells a side, z fastest,
    quotients in the particles' own precision, one last bin for the lost."""
    nb = [1 + (n + 1) // SORT_CPS for n in box.n]
    ok = None
    key = torch.zeros(x.shape, dtype=torch.int64, device=x.device)
    for p, L, m in zip((x, y, z), box.L, nb):
        width = torch.tensor(L / m, dtype=torch.float64).to(p.dtype).item()
        b = torch.floor(p / torch.full((), width, dtype=p.dtype, device=p.device)).to(torch.int64)
        inside = (b >= 0) & (b < m)
        ok = inside if ok is None else ok & inside
        key = key * m + b
    return torch.where(ok, key, torch.full_like(key, nb[0] * nb[1] * nb[2]))


# ---- state ------------------------------------------------------------------


class _View:
    """A device array of this package as torch sees it (no copy)."""

    def __init__(self, arr, shape):
        self.arr = arr
        self.__cuda_array_interface__ = {
            "shape": tuple(shape), "typestr": "<f8" if arr.dtype == np.float64 else "<f4",
            "data": (arr.ptr, False), "version": 2}


def _view(arr, shape=None):
    return torch.as_tensor(_View(arr, shape or (arr.n,)), device=DEV)


def _put(arr, t):
    """Device-to-device copy of a torch tensor into a device array."""
    t = t.contiguous()
    assert t.numel() == arr.n and t.element_size() == arr.dtype.itemsize
    torch.cuda.current_stream().synchronize()
    S._capi.check(S._capi.lib().spic_memcpy_d2d(ctypes.c_void_p(arr.ptr),
                                                ctypes.c_void_p(t.data_ptr()), arr.nbytes),
                  "copy of inputs")


class _State:
    """What a program keeps between calls; its engines end with it."""

    def __init__(self):
        self.engines, self.batch = [], None

    def __del__(self):
        if self.batch is not None:
            self.batch.close()
        for e in self.engines:
            e.close()


def _make_field(case, box, grd, seed):
    field = S.EMField(grd)
    for k, v in _field_arrays(case, box, seed).items():
        _put(field.d[k], v)
    return field


def _make_particles(case, box, s, seed):
    p = S.core.DeviceParticles(_count(case, box), _species(case, s)[0], case["prec"])
    for k, v in _particle_arrays(case, box, s, seed).items():
        _put(p.d[k], v)
    return p


def _param():
    return S.Parameters(dt=DT, c=C_LIGHT, NiterMover=3, PERIODICX=PERIODIC[0],
                        PERIODICY=PERIODIC[1], PERIODICZ=PERIODIC[2], sort_cps=SORT_CPS)


def _solve(case):
    return S.core.SolveParams(dt=DT, c=C_LIGHT, th=THETA, fourpi=FOURPI, PERIODICX=PERIODIC[0],
                              PERIODICY=PERIODIC[1], PERIODICZ=PERIODIC[2],
                              qom=[_species(case, s)[0] for s in range(case["species"])])


class _Part(S.DeviceArray):
    """A run of a larger device array, which it keeps and does not free."""

    def __init__(self, whole, first, n):
        self.whole, self.n, self.dtype = whole, n, whole.dtype
        self.nbytes = n * whole.dtype.itemsize
        self.ptr = whole.ptr + first * whole.dtype.itemsize

    def free(self):
        self.ptr = None


def _padded(n):
    return -(-n // 32) * 32


def _moment_sets(grids, block):
    """Ten moment arrays for each grid of the list; with `block`, each moment
    of all of them in one allocation, every array on a 256-byte boundary.
    Returns the sets and what a pass returns of them."""
    ids = [S.InterpDensSpecies(g) for g in grids]
    if not block:
        return ids, [[_view(i.d[n]) for n in S.MOMENT_NAMES] for i in ids]
    at = np.concatenate([[0], np.cumsum([_padded(g.nn) for g in grids])]).tolist()
    whole = {n: S.DeviceArray(at[-1], np.float64, fill_zero=True) for n in S.MOMENT_NAMES}
    for i, g, first in zip(ids, grids, at):
        i.d = {n: _Part(whole[n], first, g.nn) for n in S.MOMENT_NAMES}
    return ids, [_view(whole[n]) for n in S.MOMENT_NAMES]


def _particles_out(p):
    return {k: _view(p.d[k]) for k in COMPONENTS[:6]}


def _moment_inputs(case, box, s, seed):
    """Smooth moments with the size of the sheet's, for the field operators
    without particles."""
    g = torch.Generator(device=DEV).manual_seed(31337 * seed + s)
    rho = 0.1 / FOURPI * (-1.0 if _species(case, s)[0] < 0 else 1.0)
    uth = _species(case, s)[2]
    scale = [rho] + [rho * uth * 0.1] * 3 + [rho * uth * uth * k for k in (1, .1, .1, 1, .1, 1)]
    return [(1.0 + 0.05 * torch.randn(box.nodes, generator=g, device=DEV, dtype=torch.float64)) * a
            for a in scale]


def _vector_input(box, seed):
    g = torch.Generator(device=DEV).manual_seed(65537 * seed + 5)
    m = 3 * (box.nodes[0] - 2) * (box.nodes[1] - 2) * (box.nodes[2] - 2)
    return 1e-4 * torch.randn(m, generator=g, device=DEV, dtype=torch.float64)


def prepare(case, seed):
    S.set_async(False)
    st = _State()
    st.case = case
    st.param = _param()
    op, ns = case["op"], case["species"]
    if op == "batch":
        boxes = [_box(case, k) for k in range(case["instances"])]
        grids = [S.Grid(*box.n, *box.L, case["prec"]) for box in boxes]
        ids, st.out = _moment_sets([g for g in grids for _ in range(ns)], True)
        st.members = []
        for k, (box, grd) in enumerate(zip(boxes, grids)):
            eng = S.Engine(grd, ns)
            st.engines.append(eng)
            for s in range(ns):
                eng.load(s, _make_particles(case, box, s, seed * 64 + k))
            st.members.append((eng, _make_field(case, box, grd, seed * 64 + k),
                               ids[k * ns:(k + 1) * ns], st.param))
        st.batch = S.Batch(st.members, set_moments=True)
        return st
    box = _box(case)
    grd = st.grd = S.Grid(*box.n, *box.L, case["prec"])
    st.field = _make_field(case, box, grd, seed)
    # 64 outputs at most: the moments of more than six species in blocks
    st.ids, moments = _moment_sets([grd] * ns, ns > 6)
    st.out = {}
    if op in ("caller", "handover"):
        st.parts = [_make_particles(case, box, s, seed) for s in range(ns)]
        if case.get("calls") != "deposit":
            st.out["particles"] = [_particles_out(p) for p in st.parts]
    if op in ("phase", "handover", "cycle"):
        st.eng = S.Engine(grd, ns, set_moments=True)
        st.engines.append(st.eng)
    if op in ("phase", "cycle"):
        for s in range(ns):
            st.eng.load(s, _make_particles(case, box, s, seed))
    if op in ("cycle", "fields"):
        st.solve = _solve(case)
        st.net = S.core.InterpDensNet(grd)
        st.aux = S.core.InterpDensAux(grd)
        m = 3 * (box.nodes[0] - 2) * (box.nodes[1] - 2) * (box.nodes[2] - 2)
        st.vec = S.DeviceArray(m, np.float64)
        _put(st.vec, _vector_input(box, seed))
        st.im = S.DeviceArray(m, np.float64)
        st.out.update(rhoc=_view(st.net.rhoc), rhoh=_view(st.aux.rhoh), image=_view(st.im),
                      J=[_view(st.aux.J[k]) for k in ("Jxh", "Jyh", "Jzh")])
    if op == "fields":
        for s in range(ns):
            for name, v in zip(S.MOMENT_NAMES, _moment_inputs(case, box, s, seed)):
                _put(st.ids[s].d[name], v)
        _put(st.net.d["rhon"], sum(_moment_inputs(case, box, s, seed)[0] for s in range(ns)))
    elif not (op == "caller" and case["calls"] in ("mover", "sort")):
        st.out["moments"] = moments
    if op == "cycle":
        st.out["net"] = [_view(st.net.d[n]) for n in S.MOMENT_NAMES]
    return st


def run(st):
    case = st.case
    op, ns = case["op"], case["species"]
    if S.get_async() == case["waits"]:
        S.set_async(not case["waits"])
    if op == "caller":
        calls = case["calls"]
        for p, ids in zip(st.parts, st.ids):
            if calls in ("separate", "mover", "sort"):
                S.mover_PC(p, st.field, st.grd, st.param)
            if calls == "sort":
                S.particle_sort(st.param, p, st.grd)
            if calls in ("separate", "deposit"):
                S.setZeroSpeciesDensities([ids], st.grd, 1)
                S.interpP2G(p, ids, st.grd)
            elif calls == "fused":
                S.setZeroSpeciesDensities([ids], st.grd, 1)
                S.mover_interp(p, st.field, ids, st.grd, st.param)
    elif op == "phase":
        if case["resort"]:
            st.eng.sort()
        for _ in range(case["phases"]):
            st.eng.phase(st.field, st.ids, st.param)
    elif op == "batch":
        st.batch.phase()
    elif op == "handover":
        for s, p in enumerate(st.parts):
            st.eng.load(s, p)
        if case["push"]:
            st.eng.phase(st.field, st.ids, st.param)
        else:
            st.eng.deposit(st.ids)
        for s, p in enumerate(st.parts):
            st.eng.store(s, p)
    if op == "cycle":
        st.eng.phase(st.field, st.ids, st.param)
        S.core.applyBCids_all(st.ids, st.grd, st.param)
        S.setZeroSpeciesDensities([st.net], st.grd, 1)
        S.core.sumOverSpecies(st.net, st.ids, st.grd, ns)
    if op in ("cycle", "fields"):
        S.core.interpN2Crho_net(st.net, st.grd, st.solve)
        S.core.calculateHatDensities(st.aux, st.net, st.ids, st.field, st.grd, st.solve)
        for _ in range(case["images"]):
            S.core.MaxwellImage(st.im, st.vec, st.field, st.ids, st.grd, st.solve)
    return st.out


# ---- work -------------------------------------------------------------------


PUSH_FLOPS = 3 * (8 * 14 + 50) + 20  # three iterations of gather and rotation
DEPOSIT_FLOPS = 8 * 10 * 2 + 30


def work(case):
    w = 8 if case["prec"] == "f64" else 4
    ns = case["species"]
    op = case["op"]
    total = {"bytes": 0.0, "flops": 0.0}

    def add(b, f):
        total["bytes"] += b
        total["flops"] += f

    for k in range(case.get("instances", 1)):
        box = _box(case, k)
        nn = box.nodes[0] * box.nodes[1] * box.nodes[2]
        n = _count(case, box) * ns
        fields, moments = 6 * nn * w, 80 * nn * ns
        if op == "caller":
            calls = case["calls"]
            if calls in ("separate", "mover", "sort"):
                add(12 * w * n + fields, PUSH_FLOPS * n)
            if calls in ("separate", "deposit"):
                add(7 * w * n + moments, DEPOSIT_FLOPS * n)
            if calls == "sort":
                add(14 * w * n, 0)
            if calls == "fused":
                add(13 * w * n + fields + moments, (PUSH_FLOPS + DEPOSIT_FLOPS) * n)
        elif op == "phase":
            for _ in range(case["phases"]):
                add(13 * w * n + fields + moments, (PUSH_FLOPS + DEPOSIT_FLOPS) * n)
            if case["resort"]:
                add(14 * w * n, 0)
        elif op == "handover":
            add(13 * w * n + moments + (fields if case["push"] else 0),
                (DEPOSIT_FLOPS + (PUSH_FLOPS if case["push"] else 0)) * n)
        elif op in ("batch", "cycle"):
            add(13 * w * n + fields + moments, (PUSH_FLOPS + DEPOSIT_FLOPS) * n)
        if op == "cycle":
            add(8 * nn * (10 * ns + 10), 10 * nn * ns)
        if op in ("cycle", "fields"):
            add(8 * nn * (3 + 9 * ns + 3 + 3), 150 * nn * ns)
            for _ in range(case["images"]):
                add(8 * nn * (6 + 3 + ns), (80 + 30 * ns) * nn)
    return total


# ---- the same in 64 bits, with torch alone -----------------------------------


EXACT_MOST = 2e7  # particle steps computed below


def _cell_index(p, d, n, down):
    c = p / d
    c = torch.floor(c) if down else torch.trunc(c)
    return torch.clamp(2 + c.to(torch.int64), 1, n - 1)


def _corners(box, p, idx):
    """(node index, weight) of the eight corners of cells idx around p."""
    lo, hi = [], []
    for a in range(3):
        o = (p[a] - (idx[a] - 2).to(torch.float64) * box.d[a]) / box.d[a]
        lo.append(o)
        hi.append(1.0 - o)
    N1, N2 = box.nodes[1], box.nodes[2]
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                wgt = (lo[0] if a == 0 else hi[0]) * (lo[1] if b == 0 else hi[1]) * \
                      (lo[2] if c == 0 else hi[2])
                yield ((idx[0] - a) * N1 + idx[1] - b) * N2 + idx[2] - c, wgt


def _push64(box, f, qom, p):
    """Predictor-corrector push and particle boundary conditions."""
    x0 = [p[k] for k in "xyz"]
    v0 = [p[k] for k in "uvw"]
    pos, q2 = list(x0), qom * 0.5 * DT / C_LIGHT
    flat = [f[k].reshape(-1) for k in ("Ex", "Ey", "Ez", "Bxn", "Byn", "Bzn")]
    new = None
    for _ in range(3):
        idx = [_cell_index(pos[a], box.d[a], box.nodes[a], False) for a in range(3)]
        loc = [torch.zeros_like(x0[0]) for _ in range(6)]
        for node, wgt in _corners(box, pos, idx):
            for k in range(6):
                loc[k] += wgt * flat[k][node]
        E, B = loc[:3], loc[3:]
        t = [v0[a] + q2 * E[a] for a in range(3)]
        dot = t[0] * B[0] + t[1] * B[1] + t[2] * B[2]
        den = 1.0 / (1.0 + q2 * q2 * (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]))
        new = [(t[a] + q2 * (t[(a + 1) % 3] * B[(a + 2) % 3] - t[(a + 2) % 3] * B[(a + 1) % 3]
                             + q2 * dot * B[a])) * den for a in range(3)]
        pos = [x0[a] + new[a] * (0.5 * DT) for a in range(3)]
    for a in range(3):
        x, v, L = x0[a] + new[a] * DT, 2.0 * new[a] - v0[a], box.L[a]
        if PERIODIC[a]:
            x = torch.where(x > L, x - L, x)
            x = torch.where(x < 0, x + L, x)
        else:
            out = x > L
            x, v = torch.where(out, 2.0 * L - x, x), torch.where(out, -v, v)
            out = x < 0
            x, v = torch.where(out, -x, x), torch.where(out, -v, v)
        p["xyz"[a]], p["uvw"[a]] = x, v


def _deposit64(box, p):
    nn = box.nodes[0] * box.nodes[1] * box.nodes[2]
    inv = 1.0 / (box.d[0] * box.d[1] * box.d[2])
    pos = [p[k] for k in "xyz"]
    u, v, w, q = p["u"], p["v"], p["w"], p["q"]
    idx = [_cell_index(pos[a], box.d[a], box.nodes[a], True) for a in range(3)]
    terms = [None, u, v, w, u * u, u * v, u * w, v * v, v * w, w * w]
    out = [torch.zeros(nn, dtype=torch.float64, device=DEV) for _ in terms]
    for node, wgt in _corners(box, pos, idx):
        wgt = wgt * q * inv
        for m, t in zip(out, terms):
            m.index_add_(0, node, wgt if t is None else wgt * t)
    return out


def _ghosts64(a, nodes, zero=False):
    """Ghost planes of a scalar: periodic axes first, together; then each
    other axis from the plane inside it, or zero."""
    n = a.shape
    lo, hi = (3, 2) if nodes else (2, 1)
    idx = []
    for k in range(3):
        i = torch.arange(n[k], device=a.device)
        if PERIODIC[k]:
            i[0], i[-1] = n[k] - lo, hi
        elif not zero:
            i[0], i[-1] = 1, n[k] - 2
        idx.append(i)
    a = a[idx[0]][:, idx[1]][:, :, idx[2]].contiguous()
    if zero:
        for k in range(3):
            if not PERIODIC[k]:
                a.select(k, 0).zero_()
                a.select(k, -1).zero_()
    return a


def _d8(a, axis, inv):
    """Difference along an axis, averaged over the four pairs of corners."""
    lo, hi = a.narrow(axis, 0, a.shape[axis] - 1), a.narrow(axis, 1, a.shape[axis] - 1)
    d = (hi - lo) * inv
    for k in range(3):
        if k != axis:
            d = 0.5 * (d.narrow(k, 0, d.shape[k] - 1) + d.narrow(k, 1, d.shape[k] - 1))
    return d


def _m8(a):
    for k in range(3):
        a = 0.5 * (a.narrow(k, 0, a.shape[k] - 1) + a.narrow(k, 1, a.shape[k] - 1))
    return a


def _inner(a):
    return a[1:-1, 1:-1, 1:-1]


def _rotate64(v, om):
    dot = v[0] * om[0] + v[1] * om[1] + v[2] * om[2]
    den = 1.0 / (1.0 + om[0] ** 2 + om[1] ** 2 + om[2] ** 2)
    return [(v[a] + v[(a + 1) % 3] * om[(a + 2) % 3] - v[(a + 2) % 3] * om[(a + 1) % 3]
             + dot * om[a]) * den for a in range(3)]


def _fields64(case, box, f, net_rhon, ids, vec):
    """rhoc, hat densities and Maxwell image; ids: ten node arrays a species."""
    inv = [1.0 / d for d in box.d]
    cells = [n + 2 for n in box.n]

    def on_cells(inner):
        full = torch.zeros(cells, dtype=torch.float64, device=DEV)
        full[1:-1, 1:-1, 1:-1] = inner
        return full

    rhon = _ghosts64(net_rhon, True)
    rhoc = on_cells(_inner(_m8(rhon)))
    B = [f[k] for k in ("Bxn", "Byn", "Bzn")]
    J = [torch.zeros(box.nodes, dtype=torch.float64, device=DEV) for _ in range(3)]
    for s, m in enumerate(ids):
        P = [[m[4], m[5], m[6]], [m[5], m[7], m[8]], [m[6], m[8], m[9]]]
        beta = 0.5 * _species(case, s)[0] * DT / C_LIGHT
        om = [_inner(beta * b) for b in B]
        t = []
        for a in range(3):
            div = sum(_d8(P[k][a], k, inv[k]) for k in range(3)) * (-0.5 * DT)
            t.append(_m8(_ghosts64(on_cells(_inner(div)), False)) + _inner(m[1 + a]))
        for a, r in enumerate(_rotate64(t, om)):
            J[a][1:-1, 1:-1, 1:-1] += r
    J = [_ghosts64(j, True) for j in J]
    div = sum(_d8(J[k], k, inv[k]) for k in range(3))
    rhoh = _ghosts64(on_cells(_inner(rhoc - DT * THETA * div)), False)
    # Maxwell operator
    delt = C_LIGHT * THETA * DT
    mi = [n - 2 for n in box.nodes]
    v = vec.reshape(mi[0], mi[1], mi[2], 3)
    E = []
    for a in range(3):
        full = torch.zeros(box.nodes, dtype=torch.float64, device=DEV)
        full[1:-1, 1:-1, 1:-1] = v[..., a]
        E.append(_ghosts64(full, True, zero=True))
    D = [torch.zeros(box.nodes, dtype=torch.float64, device=DEV) for _ in range(3)]
    for s, m in enumerate(ids):
        qom = _species(case, s)[0]
        beta, coef = 0.5 * qom * DT / C_LIGHT, FOURPI / 2 * delt * DT / C_LIGHT * qom
        r = _rotate64([_inner(e) for e in E], [_inner(beta * b) for b in B])
        for a in range(3):
            D[a][1:-1, 1:-1, 1:-1] += coef * _inner(m[0]) * r[a]
    dc = _ghosts64(on_cells(_inner(sum(_d8(D[k], k, inv[k]) for k in range(3)))), False)
    im = torch.zeros_like(v)
    for a in range(3):
        e = E[a]
        lap = torch.zeros_like(_inner(e))
        for k in range(3):
            n = e.shape[k]
            sl = [slice(1, -1)] * 3
            lo, hi = list(sl), list(sl)
            lo[k], hi[k] = slice(0, n - 2), slice(2, n)
            lap = lap + (e[tuple(lo)] - 2 * _inner(e) + e[tuple(hi)]) * inv[k] ** 2
        im[..., a] = (-lap - _d8(dc, a, inv[a])) * delt * delt + _inner(D[a]) + _inner(e)
    return rhoc, rhoh, J, im.reshape(-1)


def _fold64(box, m):
    """Ghost-node fold of one moment, in place."""
    for periodic in (True, False):
        for k in range(3):
            if PERIODIC[k] != periodic:
                continue
            sl = [slice(1, -1)] * 3
            lo, hi = list(sl), list(sl)
            lo[k], hi[k] = 1, box.nodes[k] - 2
            lo, hi = tuple(lo), tuple(hi)
            if periodic:
                m[lo] += m[hi]
                m[hi] = m[lo]
            else:
                m[lo] *= 2
                m[hi] *= 2


def exact(case, seed):
    op, ns = case["op"], case["species"]
    if op == "batch":
        return None
    box = _box(case)
    n = _count(case, box)
    if op != "fields" and n * ns * case.get("phases", 1) > EXACT_MOST:
        return None
    f = {k: v.double() for k, v in _field_arrays(case, box, seed).items()}
    if op == "fields":
        ids = [_moment_inputs(case, box, s, seed) for s in range(ns)]
        rhoc, rhoh, J, im = _fields64(case, box, f, sum(i[0] for i in ids), ids,
                                      _vector_input(box, seed))
        # the net density's ghosts on the cells are not part of the result
        return {"rhoc": rhoc.reshape(-1), "rhoh": rhoh.reshape(-1), "image": im,
                "J": [j.reshape(-1) for j in J]}
    calls = case.get("calls", "")
    parts, moments = [], []
    for s in range(ns):
        p = _particle_arrays(case, box, s, seed)
        p = {k: v.double() for k, v in p.items()}
        pushes = {"caller": calls != "deposit", "handover": case.get("push", False)}.get(op, True)
        mom = None
        for _ in range(case.get("phases", 1)):
            if pushes:
                _push64(box, f, _species(case, s)[0], p)
            if calls not in ("mover", "sort"):
                mom = _deposit64(box, p)
        if calls == "sort":
            perm = torch.sort(_bins(box, p["x"], p["y"], p["z"]), stable=True).indices
            p = {k: v[perm] for k, v in p.items()}
        parts.append({k: p[k] for k in COMPONENTS[:6]})
        moments.append(mom)
    out = {}
    if op in ("caller", "handover") and calls != "deposit":
        out["particles"] = parts
        if calls == "sort" and case["prec"] == "f32":
            # a bin edge falls on either side of a rounded position
            out["particles"] = [{k: None for k in COMPONENTS[:6]} for _ in parts]
    if moments[0] is not None:
        if op == "cycle":
            moments = [[m.reshape(box.nodes) for m in ms] for ms in moments]
            for ms in moments:
                for m in ms:
                    _fold64(box, m)
            net = [sum(ms[k] for ms in moments) for k in range(10)]
            rhoc, rhoh, J, im = _fields64(case, box, f, net[0], moments, _vector_input(box, seed))
            net[0] = _ghosts64(net[0], True)
            moments = [[m.reshape(-1) for m in ms] for ms in moments]
            out.update(net=[m.reshape(-1) for m in net], rhoc=rhoc.reshape(-1),
                       rhoh=rhoh.reshape(-1), image=im, J=[j.reshape(-1) for j in J])
        if ns > 6:
            nn = moments[0][0].numel()
            pad = torch.zeros(_padded(nn) - nn, dtype=torch.float64, device=DEV)
            moments = [torch.cat([t for ms in moments for t in (ms[k], pad)]) for k in range(10)]
        out["moments"] = moments
    return out
