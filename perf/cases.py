"""The work that users have this library do, as cases to measure: whole output intervals of a
run (cycles of the drag coupling, the time step of every cycle where the run adapts it, then the
particles as the program reads them), in both forms, from a few thousand particles to a hundred
million.

A case is a dict of plain values:

  form      "fp64" (the plain form: the caller's arrays updated in place) or "fp32" (the
            cell-sorted store, exported at the end of the interval)
  box       "periodic": [0, 1)^3; "shear": the unstratified shearing box at the two-fluid
            drift equilibrium; "strat": the stratified shearing box with a continuous size
            distribution and x3 outflow; "walls": periodic in x1, x2 with reflecting x3 walls
  coupling  "imex" (imex2+, with solver "local", "dc1" or "dc2") or "pc2" (rk2)
  stencil   "tsc" or "cic"
  nx..nz    cells of a block, bx..bz blocks of the mesh per direction
  ppc       particles per cell (the mean, where block counts are uneven)
  layout    "uniform"; "clumps": half of the particles in Gaussian clumps two cells wide;
            "uneven": lognormal counts per block, uniform inside the block
  clouds    refinable clouds instead of point particles; refined: a statically refined mesh of
            three levels
  hydro     the gas moves by its own isothermal fluxes
  steps     cycles in the interval
  cycle     every cycle ends with the particles' time step (and, with x3 outflow, begins with
            the removal of the particles that left), as the reference's driver has it
  tasks     every stage driven task by task, as a task list calls the library, instead of by
            the whole-stage call
  graphs    stages run as HIP graphs on a stream of the context's own
"""

import ctypes
import math

import torch

from athenak_amd import abi, lib, workloads
from athenak_amd.lib import DustContext

DEVICE = torch.device("cuda" if torch.cuda.is_available() else "cpu")
OMEGA, QSHEAR = 1.0, 1.5
STENCIL = {"tsc": abi.DK_TSC, "cic": abi.DK_CIC}
SOLVER = {"local": abi.DK_LOCAL, "dc1": abi.DK_DC1, "dc2": abi.DK_DC2}
EXACT_MOST = 1.0e8     # particle-steps that exact() takes on (about 20 seconds)


def _case(name, form, **kw):
    c = {"form": form, "box": "periodic", "coupling": "imex", "solver": "dc1", "stencil": "tsc",
         "nx": 16, "ny": 16, "nz": 16, "bx": 1, "by": 1, "bz": 1, "ppc": 4, "layout": "uniform",
         "clouds": False, "refined": False, "hydro": False, "steps": 1, "cycle": False,
         "tasks": False, "graphs": False}
    if name:
        c["name"] = name
    if kw.get("coupling") == "pc2":
        c["solver"] = "local"
    c.update(kw)
    return c


def _cube(n, b):
    return dict(nx=n, ny=n, nz=n, bx=b, by=b, bz=b)


def listed():
    return [
        # the smallest run in earnest: a test problem or a parameter scan, where the launches
        # and the time step's round trip to the host are most of a cycle
        _case("fp64 plain box 32", "fp64", **_cube(32, 1), ppc=1, steps=1, cycle=True),
        # the same box as the FP32 form runs it between two outputs
        _case("fp32 plain box 32", "fp32", **_cube(32, 1), ppc=1, steps=20, graphs=True),
        # a production shearing box in full precision
        _case("fp64 shearing box 128", "fp64", box="shear", **_cube(64, 2), ppc=4, steps=1,
              cycle=True),
        # two-species clumping, full precision: the late state of a collapse run
        _case("fp64 clumps 64", "fp64", **_cube(32, 2), ppc=8, layout="clumps", steps=1),
        # many small blocks of very different load, the explicit coupling
        _case("fp64 pc2 uneven 64", "fp64", **_cube(16, 4), ppc=4, coupling="pc2",
              layout="uneven", steps=1),
        # a task list's own calls on a mesh of odd block sizes, two solver sweeps, walls
        _case("fp64 task list walls", "fp64", box="walls", nx=22, ny=18, nz=26, bx=2, by=3, bz=2,
              ppc=5, solver="dc2", steps=1, tasks=True),
        # the headline run: the stratified box with seven size bins per cell
        _case("fp32 stratified box 256", "fp32", box="strat", **_cube(64, 4), ppc=7, steps=6,
              cycle=True, graphs=True),
        # an ordinary shearing box
        _case("fp32 shearing box 128", "fp32", box="shear", **_cube(64, 2), ppc=4, steps=6,
              graphs=True),
        # clumps in the FP32 form
        _case("fp32 clumps 128", "fp32", **_cube(64, 2), ppc=8, layout="clumps", steps=5,
              graphs=True),
        # uneven blocks in one launch: clouds on a statically refined mesh
        _case("fp32 refined clouds", "fp32", **_cube(16, 4), ppc=4, coupling="pc2",
              layout="uneven", clouds=True, refined=True, steps=3, graphs=True),
        # uneven blocks of points
        _case("fp32 pc2 uneven 128", "fp32", **_cube(16, 8), ppc=4, coupling="pc2",
              layout="uneven", steps=8, graphs=True),
        # a dusty gas that moves by its own fluxes, one particle per cell
        _case("fp32 gas update 128", "fp32", **_cube(64, 2), ppc=1, hydro=True, steps=5,
              graphs=True),
    ]


def draw(rng):
    """One more case of the same ranges: forms, boxes, couplings and layouts as the listed
    ones mix them, block sizes with odd ones among them, particle counts spread over their
    logarithm up to 8 million (FP64) or 30 million (FP32)."""
    form = rng.choice(("fp64", "fp32"))
    kind = rng.choice(("periodic", "periodic", "clumps", "shear", "strat", "walls", "pc2", "pc2",
                       "clouds", "refined", "hydro"))
    sizes = (8, 12, 16, 20, 24, 32, 40, 48, 64)
    odd = (10, 14, 18, 22, 26, 30, 15, 21)
    if form == "fp64":
        sizes = sizes + odd
    n = [rng.choice(sizes) for _ in range(3)]
    ppc = rng.choice((1, 2, 3, 4, 5, 7, 8))
    most = 3.0e7 if form == "fp32" else 8.0e6
    target = 2.0e4*math.exp(rng.random()*math.log(most/2.0e4))
    b = [1, 1, 1]
    while b[0]*b[1]*b[2]*n[0]*n[1]*n[2]*ppc*2 <= target and b[0]*b[1]*b[2] < 512:
        d = rng.randrange(3)
        if n[d]*b[d]*2 <= 256:
            b[d] *= 2
        elif all(n[k]*b[k]*2 > 256 for k in range(3)):
            break
    while n[0]*n[1]*n[2]*b[0]*b[1]*b[2]*ppc > target and ppc > 1:
        ppc -= 1
    c = _case("", form, nx=n[0], ny=n[1], nz=n[2], bx=b[0], by=b[1], bz=b[2], ppc=ppc,
              steps=1 if form == "fp64" else rng.randint(3, 9),
              cycle=rng.random() < 0.5, graphs=form == "fp32" and rng.random() < 0.7)
    if kind in ("periodic", "shear", "walls", "strat", "clumps"):
        c["solver"] = rng.choice(("dc1", "dc1", "dc1", "dc2", "local"))
        c["stencil"] = rng.choice(("tsc", "tsc", "tsc", "cic"))
    if kind in ("shear", "strat", "walls"):
        c["box"] = kind
        if kind == "strat":
            c["ppc"] = 7 if ppc > 4 else ppc
    elif kind == "clumps":
        c["layout"] = "clumps"
    elif kind in ("pc2", "clouds", "refined"):
        c["coupling"], c["solver"] = "pc2", "local"
        c["layout"] = rng.choice(("uneven", "clumps", "uniform"))
        if kind == "clouds":
            c["clouds"] = True
        elif kind == "refined":
            c.update(clouds=True, refined=True, layout="uneven", bx=4, by=4, bz=4,
                     **dict(zip(("nx", "ny", "nz"), rng.choice(((8, 8, 8), (12, 8, 12), (16, 16, 16))))))
            if form == "fp64" or c["ppc"] > 3:
                c["ppc"] = min(c["ppc"], 3)
    elif kind == "hydro":
        c["hydro"] = True
    if form == "fp64" and not c["hydro"] and rng.random() < 0.3:
        c["tasks"] = True
    return c


# ---- the run that a case describes ---------------------------------------------------------

def _physics(c):
    shear, strat = c["box"] in ("shear", "strat"), c["box"] == "strat"
    p = abi.dk_physics(deposit=STENCIL[c["stencil"]],
                       coupling=abi.DK_PC2 if c["coupling"] == "pc2" else abi.DK_IMEX,
                       solver=SOLVER[c["solver"]], back_reaction=1, consistent_gas=1,
                       shearing_box=int(shear), stratified=int(strat), omega0=OMEGA,
                       qshear=QSHEAR, pc2_damping=0, stiffness=0, clouds=int(c["clouds"]))
    if c["coupling"] == "pc2":   # dense cells are stiff: the rate record and its damping are on
        p.pc2_damping, p.stiffness = 1, 1
    return p


def _box(c):
    return ((-0.1, 0.1),)*3 if c["box"] in ("shear", "strat") else ((0.0, 1.0),)*3


def _mesh(c):
    n, b = (c["nx"], c["ny"], c["nz"]), (c["bx"], c["by"], c["bz"])
    if c["refined"]:
        return abi.smr_mesh(n, b, _box(c), workloads.C4_REGIONS)
    return abi.uniform_mesh(
        n, b, _box(c), ng=2,
        bc_x1=abi.DK_X1_SHEAR if c["box"] in ("shear", "strat") else abi.DK_X1_PERIODIC,
        bc_x3={"strat": abi.DK_X3_OUTFLOW, "walls": abi.DK_X3_REFLECT}.get(c["box"],
                                                                           abi.DK_X3_PERIODIC))


def _source(c):
    if c["box"] in ("shear", "strat"):
        return abi.dk_gas_src(shearing_box=1, stratified=int(c["box"] == "strat"), omega0=OMEGA,
                              qshear=QSHEAR, const_accel=0.1, const_accel_dir=1)
    if c["hydro"]:
        return abi.dk_gas_src(hydro=1, iso_cs=1.0, dfloor=workloads.FLT_MIN)
    return None


def _dt(c):
    if c["hydro"]:   # a gas Courant number of 0.25
        return 0.25/max(c["nx"]*c["bx"], c["ny"]*c["by"], c["nz"]*c["bz"])
    return 2.0e-4 if c["box"] in ("shear", "strat") else 1.0e-3


def _stopping_times(c):
    """The species' stopping times and dust-to-gas ratios."""
    if c["box"] == "shear":
        return (0.1,), (3.0,)
    if c["layout"] == "clumps":
        return ((0.01, 1.0), (0.5, 0.5)) if c["coupling"] == "imex" else ((0.05,), (1.0,))
    return ((0.05,), (1.0,)) if c["coupling"] == "pc2" else ((0.1,), (1.0,))


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _counts(c, blocks, nmb, gen):
    """Particles per block."""
    cells = c["nx"]*c["ny"]*c["nz"]
    if c["layout"] != "uneven":
        return torch.full((nmb,), c["ppc"]*cells, dtype=torch.int64, device=DEVICE)
    z = torch.randn(nmb, generator=gen, device=DEVICE, dtype=torch.float64).clamp(-2.5, 2.5)
    share = torch.exp(1.5*z)
    k = torch.floor(share*(c["ppc"]*cells*nmb/float(share.sum()))).long()
    k[0] += c["ppc"]*cells*nmb - int(k.sum())   # the mean is ppc whatever the draw
    return k


def _initial(c, seed):
    """The run's initial state from the seed alone: (mesh, blocks, rdata [17, n], idata [5, n],
    the gas of the active cells [nmb, 4, nz, ny, nx])."""
    mesh, blocks = _mesh(c)
    nmb, gen = mesh.nmb, _generator(seed)
    f8 = dict(device=DEVICE, dtype=torch.float64)

    def uniform(n):
        return torch.rand(n, generator=gen, **f8)

    def normal(*n):
        return torch.randn(*n, generator=gen, **f8)

    box = _box(c)
    lo = torch.tensor([[b.x1min, b.x2min, b.x3min] for b in blocks], **f8)
    hi = torch.tensor([[b.x1max, b.x2max, b.x3max] for b in blocks], **f8)
    counts = _counts(c, blocks, nmb, gen)
    n = int(counts.sum())
    r = torch.zeros((abi.DK_NRDATA, n), **f8)
    iv = torch.zeros((abi.DK_NIDATA, n), device=DEVICE, dtype=torch.int32)
    gid = torch.repeat_interleave(torch.arange(nmb, device=DEVICE), counts)
    tag = torch.arange(n, device=DEVICE, dtype=torch.int32)
    # positions: uniform in the block
    for d, col in enumerate((abi.IPX, abi.IPY, abi.IPZ)):
        r[col] = lo[gid, d] + uniform(n)*(hi[gid, d] - lo[gid, d])
    cellw = [(box[d][1] - box[d][0])/(m*k) for d, (m, k) in
             enumerate(((c["nx"], c["bx"]), (c["ny"], c["by"]), (c["nz"], c["bz"])))]
    if c["layout"] == "clumps":   # every second particle belongs to a clump
        ncl = max(1, min(64, n//20000))
        which = torch.randint(ncl, (n,), generator=gen, device=DEVICE)
        in_clump = (tag & 1) == 1
        for d, col in enumerate((abi.IPX, abi.IPY, abi.IPZ)):
            a, b = box[d]
            x = (a + uniform(ncl)*(b - a))[which] + 2.0*cellw[d]*normal(n)
            x = a + torch.remainder(x - a, b - a)
            r[col] = torch.where(in_clump, x.clamp(max=b - 1e-9*(b - a)), r[col])
    if c["box"] == "strat":
        r[abi.IPZ] = (0.02*normal(n)).clamp(box[2][0]*0.999, box[2][1]*0.999)
    if c["layout"] == "clumps" or c["box"] == "strat":
        k = [((r[col] - box[d][0])/(box[d][1] - box[d][0])*nb).long().clamp(0, nb - 1)
             for d, (col, nb) in enumerate(((abi.IPX, c["bx"]), (abi.IPY, c["by"]),
                                            (abi.IPZ, c["bz"])))]
        gid = k[0] + c["bx"]*(k[1] + c["by"]*k[2])
    # stopping times, masses
    vol = (hi - lo).prod(1)/(c["nx"]*c["ny"]*c["nz"])
    if c["box"] == "strat":
        bin_ = (tag % 7).double()
        ts = torch.exp(math.log(1e-3) + (bin_ + uniform(n))*(math.log(1e3)/7.0))
        w = torch.sqrt(ts)
        r[abi.IPTS] = ts
        r[abi.IPM] = w*(0.01*0.2**3/float(w.sum()))
        iv[abi.PSP] = (tag % 7).int()
    else:
        taus, eps = _stopping_times(c)
        sp = (tag//2) % len(taus)
        r[abi.IPTS] = torch.tensor(taus, **f8)[sp.long()]
        r[abi.IPM] = torch.tensor(eps, **f8)[sp.long()]*len(taus)*vol[gid]/c["ppc"]
        iv[abi.PSP] = sp.int()
    # velocities
    ug = (0.0, 0.0)
    noise = 1.0e-3
    if c["box"] in ("shear", "strat"):
        noise = 1.0e-4
        taus, eps = (((0.1,), (3.0,)) if c["box"] == "shear" else ((0.1,), (0.01,)))
        ug = workloads.nsh_gas(OMEGA, QSHEAR, 0.1, eps, taus)
        t = OMEGA*r[abi.IPTS]
        r[abi.IPVX] = (ug[0] + 2.0*t*ug[1])/(1.0 + 2.0*(2.0 - QSHEAR)*t*t)
        r[abi.IPVY] = ug[1] - (2.0 - QSHEAR)*t*r[abi.IPVX]
    for col in (abi.IPVX, abi.IPVY, abi.IPVZ):
        r[col] += noise*normal(n)
    iv[abi.PGID], iv[abi.PTAG] = gid.int(), tag
    if c["refined"]:
        iv[abi.PLEV] = torch.tensor([b.level for b in blocks], device=DEVICE,
                                    dtype=torch.int32)[gid]
    # the gas
    u = torch.zeros((nmb, abi.DK_NGAS, c["nz"], c["ny"], c["nx"]), **f8)
    rho = torch.ones((nmb, c["nz"], 1, 1), **f8)
    if c["box"] == "strat":
        zc = lo[:, 2, None] + (torch.arange(c["nz"], **f8) + 0.5)*cellw[2]
        rho = torch.exp(-0.5*zc*zc)[:, :, None, None]
    u[:, 0] = rho
    if c["hydro"]:
        u[:, 0] *= 1.0 + 1.0e-3*normal(nmb, c["nz"], c["ny"], c["nx"])
    for v in range(3):
        base = ug[v] if v < 2 else 0.0
        u[:, 1 + v] = u[:, 0]*(base + noise*normal(nmb, c["nz"], c["ny"], c["nx"]))
    return mesh, blocks, r, iv, u


def prepare(case, seed):
    """What a user's program has before the interval: a context with its particles and gas
    bound (sorted once at the start of the run, as the reference's driver does)."""
    c = dict(case)
    mesh, blocks, r, iv, u = _initial(c, seed)
    n = r.shape[1]
    fp32 = c["form"] == "fp32"
    ctx = DustContext(mesh, blocks, _physics(c), n,
                      form=abi.DK_FORM_FP32 if fp32 else abi.DK_FORM_FP64,
                      stream=torch.cuda.Stream() if c["graphs"] else None)
    ctx.rdata[:, :n].copy_(r)
    ctx.idata[:, :n].copy_(iv)
    del r, iv
    g = mesh.ng
    ctx.u0[:, 0] = 1.0
    ctx.u0[:, :, g:-g, g:-g, g:-g] = u
    torch.cuda.synchronize()
    ctx.bind_particles(n)
    ctx.task("fill_gas_ghosts", abi.dk_stage(stage=1, nexp_stages=3, time=0.0, dt=0.0))
    ctx.stream.synchronize()
    ctx.u1.copy_(ctx.u0)
    torch.cuda.synchronize()
    if c["graphs"]:
        ctx.set_graphs(True)
    if not fp32:
        ctx.sort()
    torch.cuda.synchronize()
    return {"case": c, "ctx": ctx, "src": _source(c), "dt": _dt(c)}


STAGE_TASKS = ("explicit_push", "update_particle_gids", "deposit_drag", "fold_deposit_qp",
               "gas_implicit_solve", "fill_ustar", "gather_kick_pmbr", "fold_pmbr", "apply_pmbr",
               "fill_gas_ghosts")


def _task_list(ctx, dt, src):
    """One cycle through the task entries, the library's stand-in for the gas update among
    them."""
    for st in ctx.stages(dt):
        ctx.task("first_two_imp_rk", st)
        ctx._check(lib.lib().dk_gas_hook(ctx.h, ctypes.byref(st),
                                         ctypes.byref(src) if src is not None else None),
                   "gas_hook")
        ctx.task("add_drag_history_gas", st)
        for t in STAGE_TASKS:
            ctx.task(t, st)
    ctx.time += dt


def run(state):
    """One output interval, then the particles and the gas as the program reads them: the
    plain form's arrays as they lie; the FP32 form's particles in the order of their tags
    (its store is in cell order), velocities in the precision they are held in."""
    c, ctx, src = state["case"], state["ctx"], state["src"]
    ctx.stream.wait_stream(torch.cuda.current_stream())
    dt = state["dt"]
    dt_part = None
    for _ in range(c["steps"]):
        if c["cycle"] and c["box"] == "strat":
            ctx.remove_outflow_particles()
        if c["tasks"]:
            _task_list(ctx, dt, src)
        else:
            ctx.step(dt, src, check=False)
        if c["cycle"]:
            dt_part = ctx.new_time_step(0.3)
            dt = min(state["dt"], dt_part)
    g = ctx.mesh.ng
    u = ctx.u0[:, :, g:-g, g:-g, g:-g]
    if c["form"] == "fp64":
        torch.cuda.current_stream().wait_stream(ctx.stream)
        n = ctx.npart
        out = {"r": ctx.rdata[:, :n], "i": ctx.idata[:, :n], "u": u}
        if dt_part is not None:
            out["dt"] = dt_part
        return out
    ctx.export()
    n = ctx.npart
    tag, order = torch.sort(ctx.idata[abi.PTAG, :n])
    out = {"tag": tag, "x": ctx.rdata[0:6:2, :n][:, order],
           "v": ctx.rdata[1:6:2, :n].float()[:, order], "u": u}
    if dt_part is not None:
        out["dt"] = torch.tensor(dt_part, dtype=torch.float32)
    return out


def work(case):
    """Bytes and operations of an interval that its algorithm cannot do without: every stage's
    passes over the particles and the cells (each needs the mesh's result of the one before)
    with each value read and written once, and the particles written out at the end."""
    c = case
    cells = c["nx"]*c["ny"]*c["nz"]*c["bx"]*c["by"]*c["bz"]
    if c["refined"]:
        cells = c["nx"]*c["ny"]*c["nz"]*_mesh(c)[0].nmb
    n = c["ppc"]*cells
    wide = c["form"] == "fp64"
    if c["coupling"] == "pc2":
        cell = (760.0 if wide else 480.0) if c["clouds"] else (384.0 if wide else 292.0)
        part, ops = (280.0 if wide else 204.0), 27*(7 + 6 + 9)
    else:
        part, cell, ops = (648.0 if wide else 456.0), (1176.0 if wide else 732.0), 2*27*(9 + 14 + 14)
    if c["hydro"]:
        cell += 384.0
    byt = c["steps"]*(part*n + cell*cells)
    if not wide:
        byt += n*(8.0*6 + 4 + 24.0 + 12 + 4)
    if c["cycle"]:
        byt += c["steps"]*n*(40.0 if wide else 24.0)
    flops = c["steps"]*(float(ops)*n + cells*(60.0 + (900.0 if c["hydro"] else 0.0)))
    return {"bytes": byt, "flops": flops}


# ---- the same interval in plain torch, FP64 -------------------------------------------------

class _Plain:
    """The coupled stages on one global mesh with two ghost layers in x1 and x3 (x2 is periodic
    in every box)."""

    G = 2

    def __init__(self, c, mesh, r, u):
        self.c, self.r = c, r
        self.N = (c["nx"]*c["bx"], c["ny"]*c["by"], c["nz"]*c["bz"])
        self.box = _box(c)
        self.L = [b - a for a, b in self.box]
        self.dx = [self.L[d]/self.N[d] for d in range(3)]
        self.vol = self.dx[0]*self.dx[1]*self.dx[2]
        self.shear, self.strat = c["box"] in ("shear", "strat"), c["box"] == "strat"
        self.perz = c["box"] not in ("strat", "walls")
        self.u = self.to_mesh(u)
        self.u1 = self.u.clone()
        self.D = torch.zeros((3,) + self.u.shape[1:], dtype=torch.float64, device=DEVICE)
        self.time = 0.0

    def to_mesh(self, u):
        c = self.c
        v = u.reshape(c["bz"], c["by"], c["bx"], u.shape[1], c["nz"], c["ny"], c["nx"])
        return v.permute(3, 0, 4, 1, 5, 2, 6).reshape(u.shape[1], self.N[2], self.N[1],
                                                      self.N[0]).clone()

    def to_blocks(self, a):
        c = self.c
        v = a.reshape(a.shape[0], c["bz"], c["nz"], c["by"], c["ny"], c["bx"], c["nx"])
        return v.permute(1, 3, 5, 0, 2, 4, 6).reshape(-1, a.shape[0], c["nz"], c["ny"], c["nx"])

    # -- ghosts and folds
    def remap(self, col, off, eps):
        """col[..., y, x] moved by whole cells (row j from row j - off) and the fraction eps."""
        def at(s):   # the value at row j + s
            return torch.roll(col, -s, dims=-2)

        def flux(s):   # the flux through the lower face of row j + s
            b = (-2, -1, 0) if eps > 0.0 else (-1, 0, 1)
            q = [at(s + k) for k in b]
            dl, dr = q[1] - q[0], q[2] - q[1]
            p = dl*dr
            lim = torch.where(p > 0.0, 2.0*p/torch.where(p > 0.0, dl + dr, torch.ones_like(p)),
                              torch.zeros_like(p))
            return eps*(q[1] + 0.5*(1.0 - eps)*lim) if eps > 0.0 else \
                eps*(q[1] - 0.5*(1.0 + eps)*lim)
        return torch.roll(at(0) - (flux(1) - flux(0)), off, dims=-2)

    def pad(self, a, t, normal=2):
        """a with its ghosts; normal: the component that a reflecting wall negates."""
        G, (nx, ny, nz) = self.G, self.N
        p = torch.zeros((a.shape[0], nz + 2*G, ny, nx + 2*G), dtype=a.dtype, device=a.device)
        p[:, G:-G, :, G:-G] = a
        lo, hi = a[..., -G:], a[..., :G]
        if self.shear:
            ysh = QSHEAR*OMEGA*self.L[0]*t
            off, eps = int(ysh/self.dx[1]), math.fmod(ysh, self.dx[1])/self.dx[1]
            lo, hi = self.remap(lo, off, eps), self.remap(hi, -off, -eps)
        p[:, G:-G, :, :G], p[:, G:-G, :, -G:] = lo, hi
        for g in range(G):
            if self.perz:
                p[:, g], p[:, -1 - g] = p[:, nz + g], p[:, 2*G - 1 - g]
            else:
                refl = self.c["box"] == "walls"
                p[:, G - 1 - g] = p[:, G + g] if refl else p[:, G]
                p[:, nz + G + g] = p[:, nz + G - 1 - g] if refl else p[:, nz + G - 1]
                if refl:
                    p[normal, G - 1 - g] *= -1.0
                    p[normal, nz + G + g] *= -1.0
        return p

    def fold(self, p, t):
        """The active part of p with its ghosts' sums added where they belong."""
        G, (nx, ny, nz) = self.G, self.N
        p = p.clone()
        for g in range(G):
            if self.perz:
                p[:, nz + g] += p[:, g]
                p[:, 2*G - 1 - g] += p[:, -1 - g]
            else:
                p[:, G + g] += p[:, G - 1 - g]
                p[:, nz + G - 1 - g] += p[:, nz + G + g]
        p = p[:, G:-G]
        a, lo, hi = p[..., G:-G].clone(), p[..., :G], p[..., -G:]
        if self.shear:
            s = math.fmod(QSHEAR*OMEGA*self.L[0]*t, self.L[1])/self.dx[1]

            def moved(q, sh):
                k = math.floor(sh)
                return (1.0 - (sh - k))*torch.roll(q, k, dims=-2) + \
                    (sh - k)*torch.roll(q, k + 1, dims=-2)
            lo, hi = moved(lo, -s), moved(hi, s)
        a[..., -G:] += lo
        a[..., :G] += hi
        return a

    # -- particles and mesh
    def stencil(self, x, y, z):
        out = []
        for d, q in enumerate((x, y, z)):
            s = (q - self.box[d][0])/self.dx[d]
            i = torch.floor(s)
            e = s - (i + 0.5)
            w = ((0.5*(0.5 - e)**2, 0.75 - e*e, 0.5*(0.5 + e)**2) if self.c["stencil"] == "tsc"
                 else ((-e).clamp(min=0.0), 1.0 - e.abs(), e.clamp(min=0.0)))
            out.append((i.long(), w, e))
        return out

    def cells(self, st):
        """(flat padded index, weight, the offsets) of the 27 cells."""
        G, (nx, ny, nz) = self.G, self.N
        for k in range(3):
            for j in range(3):
                row = (torch.remainder(st[1][0] + (j - 1), ny))
                plane = (st[2][0] + (k - 1 + G)).clamp(0, nz + 2*G - 1)
                for i in range(3):
                    col = (st[0][0] + (i - 1 + G)).clamp(0, nx + 2*G - 1)
                    yield ((plane*ny + row)*(nx + 2*G) + col, st[2][1][k]*st[1][1][j]*st[0][1][i],
                           (i, j, k))

    def gather(self, p, st):
        f = p.reshape(p.shape[0], -1)
        out = torch.zeros((p.shape[0], st[0][0].numel()), dtype=p.dtype, device=p.device)
        for idx, w, _ in self.cells(st):
            for v in range(f.shape[0]):
                out[v] += w*f[v][idx]
        return out

    def gather_cloud(self, p, st):
        """The linear gather of a cloud of half-width one cell."""
        def moment(s):
            s = s.clamp(-1.0, 1.0)
            return 0.5*s*s - s.abs()**3/3.0
        h = [[moment(a - 0.5 - e) - moment(a - 1.5 - e) for a in range(3)] for _, _, e in st]
        q = [p]
        for dim in (3, 2, 1):
            q.append(torch.roll(p, -1, dims=dim) - torch.roll(p, 1, dims=dim))
        q = [t.reshape(3, -1) for t in q]
        out = torch.zeros((3, st[0][0].numel()), dtype=p.dtype, device=p.device)
        for idx, w, (i, j, k) in self.cells(st):
            wx, wy, wz = st[0][1][i], st[1][1][j], st[2][1][k]
            cx = 0.5*(wy*wz*h[0][i] + (st[0][2] + (1 - i))*w)
            cy = 0.5*(wx*wz*h[1][j] + (st[1][2] + (1 - j))*w)
            cz = 0.5*(wx*wy*h[2][k] + (st[2][2] + (1 - k))*w)
            for v in range(3):
                out[v] += w*q[0][v][idx] + cx*q[1][v][idx] + cy*q[2][v][idx] + cz*q[3][v][idx]
        return out

    def deposit(self, vals, st, t):
        G, (nx, ny, nz) = self.G, self.N
        p = torch.zeros((len(vals), (nz + 2*G)*ny*(nx + 2*G)), dtype=torch.float64, device=DEVICE)
        for idx, w, _ in self.cells(st):
            for v, q in enumerate(vals):
                p[v].index_add_(0, idx, w*q)
        return self.fold(p.reshape(len(vals), nz + 2*G, ny, nx + 2*G), t)

    # -- the gas update
    def flux_divergence(self, cs=1.0):
        w = self.u.clone()
        w[1:] /= w[0]
        out = torch.zeros_like(w)
        for d, dim in enumerate((3, 2, 1)):
            order = [0] + [1 + (d + k) % 3 for k in range(3)]
            q = w[order]

            def at(a, s):
                return torch.roll(a, -s, dims=dim)
            dl, dr = q - at(q, -1), at(q, 1) - q
            p = dl*dr
            lim = torch.where(p > 0.0, p/torch.where(p > 0.0, dl + dr, torch.ones_like(p)),
                              torch.zeros_like(p))
            wl, wr = at(q + lim, -1), q - lim     # the states of each cell's lower face
            sl, sr = torch.sqrt(wl[0]), torch.sqrt(wr[0])
            vroe = (sl*wl[1] + sr*wr[1])/(sl + sr)
            bp = torch.maximum(vroe + cs, wr[1] + cs)
            bm = torch.minimum(vroe - cs, wl[1] - cs)
            bp = torch.where(bp > 0.0, bp, torch.full_like(bp, 1e-20))
            bm = torch.where(bm < 0.0, bm, torch.full_like(bm, -1e-20))
            fl, fr = wl[0]*(wl[1] - bm), wr[0]*(wr[1] - bp)
            fl = torch.stack([fl] + [wl[k]*fl for k in (1, 2, 3)])
            fr = torch.stack([fr] + [wr[k]*fr for k in (1, 2, 3)])
            fl[1] += cs*cs*wl[0]
            fr[1] += cs*cs*wr[0]
            f = 0.5*(fl + fr) + 0.5*(bp + bm)/(bp - bm)*(fl - fr)
            out[order] += (at(f, 1) - f)/self.dx[d]
        return out

    def gas_update(self, g0, g1, bdt):
        rho, m = self.u[0].clone(), self.u[1:].clone()
        new = g0*self.u + g1*self.u1
        if self.c["hydro"]:
            new -= bdt*self.flux_divergence()
        if self.shear:
            new[1] += bdt*0.1*rho + 2.0*bdt*OMEGA*m[1]
            new[2] -= (2.0 - QSHEAR)*bdt*OMEGA*m[0]
            if self.strat:
                z = self.box[2][0] + (torch.arange(self.N[2], device=DEVICE,
                                                   dtype=torch.float64) + 0.5)*self.dx[2]
                new[3] -= bdt*OMEGA*OMEGA*rho*z[:, None, None]
        self.u = new

    # -- migration
    def migrate(self, ysh, dsh):
        r = self.r
        if not self.perz:
            a, b = self.box[2]
            low, high = r[abi.IPZ] < a, r[abi.IPZ] >= b
            out = low | high
            zf = torch.where(low, torch.full_like(r[0], a), torch.full_like(r[0], b))
            if self.c["box"] == "walls":
                z = (2.0*zf - r[abi.IPZ]).clamp(min=a, max=b - 1e-12*(b - a))
                r[abi.IPZ] = torch.where(out, z, r[abi.IPZ])
                r[abi.IPZ1] = torch.where(out, 2.0*zf - r[abi.IPZ1], r[abi.IPZ1])
                for col in (abi.IPVZ, abi.IPVZ1):
                    r[col] = torch.where(out, -r[col], r[col])
            else:
                half = 0.5*self.dx[2]
                z = torch.where(low, zf + half, zf - half)
                zero = torch.zeros_like(z)
                r[abi.IPM] = torch.where(out, zero, r[abi.IPM])
                r[abi.IPZ] = torch.where(out, z, r[abi.IPZ])
                for col in (abi.IPVX, abi.IPVY, abi.IPVZ, abi.IPVX1, abi.IPVY1, abi.IPVZ1):
                    r[col] = torch.where(out, zero, r[col])
                for col in (abi.IPX, abi.IPY, abi.IPZ):
                    r[col + 6] = torch.where(out, r[col], r[col + 6])
        for d, col in enumerate((abi.IPX, abi.IPY, abi.IPZ)):
            a, b = self.box[d]
            low, high = r[col] < a, r[col] >= b
            k = low.double() - high.double()
            r[col] += k*(b - a)
            r[col + 6] += k*(b - a)
            if d == 0 and self.shear:
                y = r[abi.IPY] - k*(ysh + dsh)
                r[abi.IPY1] += y - r[abi.IPY]
                r[abi.IPY] = y

    def store(self, cols, vals):
        for col, v in zip(cols, vals):
            self.r[col] = v

    def imex(self, dt):
        r, X, V = self.r, (abi.IPX, abi.IPY, abi.IPZ), (abi.IPVX, abi.IPVY, abi.IPVZ)
        R = (abi.IPRX, abi.IPRY, abi.IPRZ)
        for st in abi.imex2p_stages(self.time, dt)[:2]:
            s = st.stage - 1
            g0, g1, bdt, a = st.gam0[s], st.gam1[s], st.beta[s]*dt, st.a_impl*dt
            atw = st.a_twid22*dt if s == 1 else 0.0
            if s == 0:
                self.u1 = self.u.clone()
                for col in X + V:
                    r[col + 6] = r[col]
            self.gas_update(g0, g1, bdt)
            self.u[1:] += atw*self.D
            old = [r[k].clone() for k in X + V]
            f = [0.0, 0.0, 0.0]
            ydot = old[4]
            if self.shear:
                f = [2.0*OMEGA*old[4], -(2.0 - QSHEAR)*OMEGA*old[3],
                     -OMEGA*OMEGA*old[2] if self.strat else 0.0]
                ydot = old[4] - QSHEAR*OMEGA*old[0]
            for d in range(3):
                r[V[d]] = g0*old[3 + d] + g1*r[V[d] + 6] + bdt*f[d] + atw*r[R[d]]
                r[X[d]] = g0*old[d] + g1*r[X[d] + 6] + bdt*(ydot if d == 1 else old[3 + d])
            ysh = dsh = sh = 0.0
            if self.shear:
                w = 0.0
                for k in range(st.stage + 1, st.nexp_stages + 1):
                    w = st.gam0[k - 1]*w + st.beta[k - 1]
                cc = 0.0
                for k in range(st.stage):
                    cc = st.gam0[k]*cc + st.beta[k]
                ysh = math.fmod(QSHEAR*OMEGA*self.L[0]*self.time, self.L[1])
                dsh = QSHEAR*OMEGA*self.L[0]*(1.0 - w)*dt
                sh = QSHEAR*OMEGA*cc*dt
            self.migrate(ysh, dsh)
            x, v = [r[k] for k in X], torch.stack([r[k] for k in V])
            at = self.stencil(x[0], x[1] + sh*x[0], x[2])
            cj = a/(r[abi.IPTS] + a)
            muc = r[abi.IPM]*cj/self.vol
            q = self.deposit([muc] + [muc*v[d] for d in range(3)], at, self.time)
            rho, b = self.u[0], self.u[1:] + q[1:]
            us = b/(rho + q[0])
            for _ in range({"local": 0, "dc1": 1, "dc2": 2}[self.c["solver"]]):
                g = self.gather(self.pad(us, self.time), at)
                au = self.deposit([muc*g[d] for d in range(3)], at, self.time) + rho*us
                us = us + (b - au)/(rho + q[0])
            dv = cj*(self.gather(self.pad(us, self.time), at) - v)
            v = v + dv
            rate = dv/a
            fac = -r[abi.IPM]/self.vol
            D = self.deposit([fac*dv[d] for d in range(3)], at, self.time)
            own = self.stencil(*x)
            inside = [own[d][0].clamp(0, self.N[d] - 1) for d in range(3)]
            flat = (inside[2]*self.N[1] + inside[1])*self.N[0] + inside[0]
            qt = torch.zeros(rho.numel(), dtype=torch.float64, device=DEVICE)
            qt.index_add_(0, flat, muc)
            qt = qt.reshape(rho.shape)
            gg = rho*us - self.u[1:]
            rr = (D - gg)/(rho + q[0])
            some = qt > 0.0
            dgas = torch.where(some, gg + rho*rr, D)
            res = torch.where(some, rr*q[0]/torch.where(some, qt, torch.ones_like(qt)),
                              torch.zeros_like(rr))
            self.u[1:] += dgas
            self.D = dgas/a
            live = r[abi.IPM] > 0.0
            for d in range(3):
                c = torch.where(live, cj*res[d].reshape(-1)[flat], torch.zeros_like(cj))
                r[V[d]] = v[d] + c
                r[R[d]] = rate[d] + c/a
        self.time += dt

    def pc2(self, dt):
        r, X, V = self.r, (abi.IPX, abi.IPY, abi.IPZ), (abi.IPVX, abi.IPVY, abi.IPVZ)
        gather = self.gather_cloud if self.c["clouds"] else self.gather
        self.u1 = self.u.clone()
        for col in X + V:
            r[col + 6] = r[col]
        self.gas_update(0.0, 1.0, dt)
        at = self.stencil(*[r[k] for k in X])
        ug = gather(self.pad(self.u1[1:]/self.u1[0], self.time), at)
        rate = r[abi.IPM]/(r[abi.IPTS]*self.vol)
        g = self.deposit([-dt*rate*(ug[d] - r[V[d]]) for d in range(3)] + [rate], at, self.time)
        chi = dt*g[3]/self.u[0]
        g = torch.where(chi > 1.0, g[:3]/chi.clamp(min=1.0), g[:3])
        self.u[1:] += g
        us = (self.u1[1:] + self.u[1:])/(self.u1[0] + self.u[0])
        self.gas_update(0.5, 0.5, 0.5*dt)
        x0, v0 = [r[k].clone() for k in X], [r[k].clone() for k in V]
        xh = [x0[d] + 0.5*dt*v0[d] for d in range(3)]
        at = self.stencil(*[self.box[d][0] + torch.remainder(xh[d] - self.box[d][0], self.L[d])
                            for d in range(3)])
        ug = gather(self.pad(us, self.time), at)
        lam = 0.5*dt/r[abi.IPTS]
        vh = [(v0[d] + lam*ug[d])/(1.0 + lam) for d in range(3)]
        dv = [dt*(ug[d] - vh[d])/r[abi.IPTS] for d in range(3)]
        self.store(V, [2.0*vh[d] - v0[d] for d in range(3)])
        self.store(X, [x0[d] + dt*vh[d] for d in range(3)])
        self.store([k + 6 for k in X], xh)
        self.store((abi.IPRX, abi.IPRY, abi.IPRZ), dv)
        fac = -r[abi.IPM]/self.vol
        self.u[1:] += self.deposit([fac*dv[d] for d in range(3)], at, self.time) - 0.5*g
        self.migrate(0.0, 0.0)
        self.time += dt

    def time_step(self, cfl):
        r = self.r
        v = [r[abi.IPVX], r[abi.IPVY], r[abi.IPVZ]]
        if self.shear:
            v[1] = v[1] - QSHEAR*OMEGA*r[abi.IPX]
        dt = cfl*min(self.dx[d]/max(float(v[d].abs().max()), 1e-30) for d in range(3))
        if self.shear and self.c["form"] == "fp32":   # the FP32 form's frame-shift limit
            cmax = 1.0 + math.sqrt(0.5)
            dt = min(dt, (1.0 - 1e-9)*0.5*self.dx[1]/(QSHEAR*OMEGA*cmax*0.1))
        return dt


def exact(case, seed):
    """The interval's outputs in plain torch, 64 bits.  None on a refined mesh (a traversal of
    leaves of several levels per cloud) and for runs that would take too long."""
    c = dict(case)
    n = c["ppc"]*c["nx"]*c["ny"]*c["nz"]*c["bx"]*c["by"]*c["bz"]
    if c["refined"] or n*c["steps"] > EXACT_MOST:
        return None
    mesh, blocks, r, iv, u = _initial(c, seed)
    fp64 = c["form"] == "fp64"
    if fp64:   # the plain form's arrays in the order of its sort by block and cell
        cell = []
        for d, (col, m, k) in enumerate(((abi.IPX, c["nx"], c["bx"]), (abi.IPY, c["ny"], c["by"]),
                                         (abi.IPZ, c["nz"], c["bz"]))):
            lo = torch.tensor([(b.x1min, b.x2min, b.x3min)[d] for b in blocks],
                              dtype=torch.float64, device=DEVICE)
            hi = torch.tensor([(b.x1max, b.x2max, b.x3max)[d] for b in blocks],
                              dtype=torch.float64, device=DEVICE)
            g = iv[abi.PGID].long()
            cell.append((((r[col] - lo[g])*(m/(hi[g] - lo[g])) + 1.0).long() - 1))
        key = ((iv[abi.PGID].long()*c["nz"] + cell[2])*c["ny"] + cell[1])*c["nx"] + cell[0]
        order = torch.sort(key, stable=True)[1]
        r = r[:, order].clone()
    sim = _Plain(c, mesh, r, u)
    dt, dt_part = _dt(c), None
    for _ in range(c["steps"]):
        if c["cycle"] and c["box"] == "strat":
            sim.r = sim.r[:, sim.r[abi.IPM] != 0.0].clone()
        (sim.pc2 if c["coupling"] == "pc2" else sim.imex)(dt)
        if c["cycle"]:
            dt_part = sim.time_step(0.3)
            dt = min(_dt(c), dt_part)
    gas = sim.to_blocks(sim.u)
    if fp64:
        out = {"r": sim.r, "i": None, "u": gas}
    else:
        out = {"tag": None, "x": sim.r[0:6:2], "v": sim.r[1:6:2], "u": gas}
    if dt_part is not None:
        out["dt"] = dt_part
    return out
