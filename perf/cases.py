"""Performance cases: the work a user of spade_amd has it do, through the
public Python entry points (which mirror the C ABI one to one).

Five operations, over small, ordinary and large grids, block shapes that
divide into nothing in particular, both coordinate kinds and both residual
modes:

  rhs    flux_div on a resident array (the residual a user's own time loop
         or a callback asks for);
  host   a SPADE-side adapter call: primitives in host memory, upload,
         ghost exchange, flux_div, residual back in host memory;
  ssprk3 Integrator.advance(steps), the library's own stepping; with
         ``monitor`` also the CFL wave speed and the kinetic-energy /
         enstrophy diagnostics a run prints every few steps;
  rk4    RKIntegrator with a general Butcher table and the default residual
         and boundary step;
  batch  Batch.step(steps) of an ensemble of periodic cases, with the
         per-case histories a study or the serving loop collects.

Arrays live on the device behind handles.  What ``run`` returns are those
arrays: ``Arrays`` reads one from the device (``download``, the reference's
host layout) when it is looked up, so a pass ends where a user's program
would go on with the array, not with a copy across PCIe.  In the ``host``
case the copies are part of the call and of the pass.

``exact`` evaluates the same formulas in plain torch, FP64, on the whole
(unblocked) grid.
"""
import math

import numpy as np
import torch

import spade_amd as sa

GAMMA, PRANDTL, POWER = 1.4, 0.72, 0.76
TANH_BETA, T_WALL = 1.5, 1.0
NG = 2                          # ghost layers
P, T, U, V, W = range(5)        # primitive order

# flux compositions: what the repository's benchmark, studies and golden tests
# compose.  mach / mu set the flow they are run on.
#   keep2_visc        the Taylor-Green headline (power-law viscosity)
#   keep2_pdiss_visc  the channel's (constant sensor, power law)
#   keep2_ducros_visc the same with the Ducros sensor and constant viscosity
#   keep4_wale        large-eddy simulation: fourth-order KEEP, WALE subgrid
#   weno_visc, fweno_visc  shock capturing
#   totani_visc       the low-cost split form
FLUXES = {
    "keep2_visc": dict(mach=0.1, mu=1.0 / 1600.0, flops=600),
    "keep2_pdiss_visc": dict(mach=0.2, mu=1.0 / 2800.0, flops=750),
    "keep2_ducros_visc": dict(mach=0.3, mu=1.0e-3, flops=800),
    "keep4_wale": dict(mach=0.2, mu=1.0 / 5000.0, flops=1300),
    "weno_visc": dict(mach=0.5, mu=1.0e-3, flops=2000),
    "fweno_visc": dict(mach=0.5, mu=1.0e-3, flops=1500),
    "totani_visc": dict(mach=0.1, mu=1.0 / 1600.0, flops=700),
}


def _case(name, op, cells, blocks, flux="keep2_visc", stretch=False, increment=False, steps=1, monitor=False):
    c = dict(op=op, cx=cells[0], cy=cells[1], cz=cells[2], bx=blocks[0], by=blocks[1], bz=blocks[2], flux=flux,
             stretch=stretch, increment=increment, steps=steps, monitor=monitor)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: the golden tests' rough periodic grid, all launch and host latency
        _case("rhs_small", "rhs", (4, 8, 4), (2, 3, 2)),
        # the headline: one residual of the 256^3 Taylor-Green vortex in 16^3 blocks
        _case("rhs_tgv_256", "rhs", (16, 16, 16), (16, 16, 16)),
        # the wall-bounded channel on stretched coordinates, 192 x 128 x 96
        _case("rhs_channel", "rhs", (16, 16, 16), (12, 8, 6), "keep2_pdiss_visc", stretch=True),
        # a mesh whose blocks are not 16 wide (users cut domains to fit, not to tile)
        _case("rhs_ragged", "rhs", (24, 20, 12), (5, 6, 8)),
        # shock capturing on the 128^3 grid of the compositions benchmark
        _case("rhs_weno_128", "rhs", (16, 16, 16), (8, 8, 8), "weno_visc"),
        # large-eddy residual added to a source already in rhs, few big blocks
        _case("rhs_les_96", "rhs", (32, 32, 32), (3, 3, 3), "keep4_wale", increment=True),
        # the CPU-sized Taylor-Green run: 64^3, ten steps to a call
        _case("step_tgv_64", "ssprk3", (16, 16, 16), (4, 4, 4), steps=10),
        # the full-size run: 256^3, a few steps between outputs
        _case("step_tgv_256", "ssprk3", (16, 16, 16), (16, 16, 16), steps=4),
        # the channel as it is run: steps with walls, then wave speed and diagnostics
        _case("step_channel", "ssprk3", (16, 16, 16), (12, 8, 6), "keep2_pdiss_visc", stretch=True, steps=10,
              monitor=True),
        # a general Butcher table, shock capturing, walls, stretched, odd blocks
        _case("rk4_weno_walls", "rk4", (20, 12, 16), (4, 4, 4), "weno_visc", stretch=True, steps=2),
        # the batched engine: an ensemble in one pool, a serving round's few steps
        dict(name="ensemble_60", op="batch", n=60, pick=7, lo=32, hi=96, steps=4),
        # a host program that keeps its arrays and offloads the residual, 64^3
        _case("host_rhs_64", "host", (16, 16, 16), (4, 4, 4)),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    op = rng.choice(["rhs", "rhs", "rhs", "rhs", "ssprk3", "ssprk3", "rk4", "batch", "host"])
    if op == "batch":
        return dict(op="batch", n=int(_log(rng, 2, 60)), pick=rng.randrange(1, 1000), lo=32,
                    hi=rng.choice([48, 64, 96]), steps=rng.randrange(1, 5))
    flux = rng.choice(sorted(FLUXES) + ["keep2_visc", "keep2_pdiss_visc"])
    # cells: up to the headline's for the cheap residual, less where a pass is
    # many residuals, a heavier flux or copies across PCIe
    most = {"rhs": 16.7e6, "ssprk3": 8.0e6, "rk4": 1.0e6, "host": 2.0e6}[op]
    if flux not in ("keep2_visc", "keep2_pdiss_visc"):
        most = min(most, 2.0e6)
    steps = 1 if op in ("rhs", "host") else rng.randrange(1, 4)
    stretch = rng.random() < 0.35
    if rng.random() < 0.4:
        cells = (16, 16, 16)
    else:
        cells = tuple(int(round(_log(rng, 4, 40))) for _ in range(3))
    if cells != (16, 16, 16) or flux not in ("keep2_visc", "keep2_pdiss_visc", "keep2_ducros_visc"):
        # a residual outside the library's tuned set can cost some 2 ns a cell,
        # 4 on stretched coordinates, more in blocks narrower than a wavefront's
        # rows: keep a pass below the largest listed one
        idle = (math.ceil(cells[0] / 16) * 16 / cells[0]) * (math.ceil(cells[1] / 4) * 4 / cells[1])
        residuals = steps * {"ssprk3": 3, "rk4": 4}.get(op, 1)
        most = min(most, 7.0e-3 / ((4.0e-9 if stretch else 2.0e-9) * idle * residuals))
    want = max(1.0, _log(rng, 4.0e3, max(most, 8.0e3)) / (cells[0] * cells[1] * cells[2]))
    blocks = [1, 1, 1]
    while blocks[0] * blocks[1] * blocks[2] < want:
        # grow the shortest axis, now and then another one
        a = rng.randrange(3) if rng.random() < 0.3 else min(range(3), key=lambda d: blocks[d] * cells[d])
        blocks[a] += 1
        if cells[0] * cells[1] * cells[2] * blocks[0] * blocks[1] * blocks[2] > most:
            blocks[a] = max(1, blocks[a] - 1)
            break
    return _case(None, op, cells, blocks, flux, stretch=stretch,
                 increment=op == "rhs" and rng.random() < 0.25, steps=steps,
                 monitor=op == "ssprk3" and rng.random() < 0.3)


# ---------------------------------------------------------------- the flow ---

def _flow(case):
    """Gas, viscosity and domain of a grid case."""
    f = FLUXES[case["flux"]]
    c0 = 1.0 / f["mach"]
    R = c0 * c0 / GAMMA                         # rho0 = T0 = u0 = 1
    if case["stretch"]:
        lo, hi = (0.0, -1.0, 0.0), (4.0 * math.pi, 1.0, 4.0 * math.pi / 3.0)
    else:
        lo, hi = (0.0, 0.0, 0.0), (2.0 * math.pi,) * 3
    n = (case["cx"] * case["bx"], case["cy"] * case["by"], case["cz"] * case["bz"])
    dx = [(hi[a] - lo[a]) / n[a] for a in range(3)]
    dmin = min(dx)
    if case["stretch"]:
        t = math.tanh(TANH_BETA * (1.0 - 0.5 * dx[1]))
        dmin = min(dx[0], dx[2], dx[1] * TANH_BETA * (1.0 - t * t) / math.tanh(TANH_BETA))
    dt = 0.4 * dmin / (1.7 + c0)
    # explicit viscous limit on the finest cell
    dt = min(dt, 0.1 * dmin * dmin / (6.0 * f["mu"]))
    return dict(f, R=R, p0=R, lo=lo, hi=hi, n=n, dx=dx, dt=dt)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _interior(case, seed):
    """Primitives on the whole grid, (5, nz, ny, nx): a Taylor-Green vortex
    with seeded phases, or a Poiseuille profile between walls, plus small
    seeded fluctuations of every variable."""
    f, dev = _flow(case), _device()
    g = torch.Generator(device=dev).manual_seed(int(seed) * 7919 + 13)
    ph = torch.rand(3, generator=g, device=dev, dtype=torch.float64).tolist()
    nx, ny, nz = f["n"]
    x, y, z = (f["lo"][a] + (torch.arange(f["n"][a], device=dev, dtype=torch.float64) + 0.5) * f["dx"][a]
               for a in range(3))
    x, y, z = x.view(1, 1, nx), y.view(1, ny, 1), z.view(nz, 1, 1)
    q = torch.rand((5, nz, ny, nx), generator=g, device=dev, dtype=torch.float64).sub_(0.5)
    q[P] *= 2e-4 * f["p0"]
    q[T] *= 2e-3
    q[U:] *= 0.05
    q[P] += f["p0"]
    q[T] += 1.0
    if case["stretch"]:
        yy = torch.tanh(TANH_BETA * y) / math.tanh(TANH_BETA)
        q[U] += 1.5 * (1.0 - yy * yy)
        q[V] += 0.02 * torch.sin(x + 6.0 * ph[0]) * (1.0 - yy * yy)
    else:
        a, b, c = (x + 6.0 * ph[0], y + 6.0 * ph[1], z + 6.0 * ph[2])
        q[U] += torch.sin(a) * torch.cos(b) * torch.cos(c)
        q[V] -= torch.cos(a) * torch.sin(b) * torch.cos(c)
        q[P] += (torch.cos(2 * a) + torch.cos(2 * b)) * (torch.cos(2 * c) + 2.0) / 16.0
    return q


def _pad(case, q):
    """q with its NG ghost layers: periodic axes wrap, and between walls (y)
    the no-slip isothermal mirror of the cells, x- and z-ghosts included."""
    def wrap(a, d):
        n = a.shape[d]
        return torch.cat([a.narrow(d, n - NG, NG), a, a.narrow(d, 0, NG)], d)
    q = wrap(wrap(q, 1), 3)
    if not case["stretch"]:
        return wrap(q, 2)

    def mirror(part):
        m = -part.flip(2)
        m[P] = -m[P]
        m[T] += 2.0 * T_WALL
        return m
    return torch.cat([mirror(q.narrow(2, 0, NG)), q, mirror(q.narrow(2, q.shape[2] - NG, NG))], 2)


def _to_blocks(case, padded):
    """A padded whole-grid field as the host image: (blocks, Nz, Ny, Nx, 5)."""
    b = padded
    for d, c in ((1, "cz"), (2, "cy"), (3, "cx")):
        b = b.unfold(d, case[c] + 2 * NG, case[c])
    b = b.permute(1, 2, 3, 4, 5, 6, 0)
    return b.reshape(-1, *b.shape[3:]).contiguous()


def _ghostless(case, q):
    """An interior whole-grid field as a host image with zero ghosts."""
    nz, ny, nx = q.shape[1:]
    b = q.reshape(5, case["bz"], case["cz"], case["by"], case["cy"], case["bx"], case["cx"])
    b = b.permute(1, 3, 5, 2, 4, 6, 0).reshape(-1, case["cz"], case["cy"], case["cx"], 5)
    return torch.nn.functional.pad(b, (0, 0, NG, NG, NG, NG, NG, NG))


def _source(case, seed):
    """What is in rhs before an incrementing residual."""
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(int(seed) * 104729 + 5)
    nx, ny, nz = _flow(case)["n"]
    return torch.rand((5, nz, ny, nx), generator=g, device=dev, dtype=torch.float64)


# ----------------------------------------------------------- prepare / run ---

class Arrays(dict):
    """Device arrays of a state by name; looking one up reads it from the
    device (the state that owns them lives as long as this does)."""

    def __init__(self, owner, **arrays):
        super().__init__(**arrays)
        self.owner = owner

    def __getitem__(self, key):
        v = dict.__getitem__(self, key)
        return v.download() if isinstance(v, sa.GridArray) else v


class State:
    """The objects a user's program keeps for one case."""

    def __init__(self):
        self.keep = []

    def add(self, obj):
        self.keep.append(obj)
        return obj

    def __del__(self):
        for obj in reversed(self.keep):
            obj.close()


def _flux(case, gas):
    f, name = FLUXES[case["flux"]], case["flux"]
    power = sa.power_law(f["mu"], 1.0, POWER, PRANDTL)
    const = sa.constant_viscosity(f["mu"], PRANDTL)
    if name == "keep2_visc":
        return sa.compose(sa.cent_keep(2, gas), sa.visc_lr(power, gas))
    if name == "keep2_pdiss_visc":
        return sa.compose(sa.cent_keep(2, gas), sa.pressure_diss_lr(gas, sa.const_sensor(0.5), 0.1, 0.1),
                          sa.visc_lr(power, gas))
    if name == "keep2_ducros_visc":
        return sa.compose(sa.cent_keep(2, gas), sa.pressure_diss_lr(gas, sa.ducros(1e-2), 0.1, 0.05),
                          sa.visc_lr(const, gas))
    if name == "keep4_wale":
        return sa.compose(sa.cent_keep(4, gas), sa.visc_lr(sa.sgs_visc(power, sa.wale(gas, 0.5, 0.06, 0.9)), gas))
    if name == "weno_visc":
        return sa.compose(sa.weno(gas), sa.visc_lr(const, gas))
    if name == "fweno_visc":
        return sa.compose(sa.fweno(gas), sa.visc_lr(const, gas))
    return sa.compose(sa.totani_lr(gas), sa.visc_lr(power, gas))


def _specs(case, seed):
    """The ensemble's cases: sizes and kinds from the case, Mach and Reynolds
    numbers from the seed."""
    import random
    sizes, flow = random.Random(case["pick"]), random.Random(int(seed))
    axis = [c for c in (32, 48, 64, 96) if case["lo"] <= c <= case["hi"]]
    out = []
    for _ in range(case["n"]):
        kind = sizes.choice(["tgv", "vortex"])
        cells = tuple(sizes.choice(axis) for _ in range(3))
        out.append(sa.CaseSpec(kind, cells, mach=flow.uniform(0.1, 0.4), reynolds=_log(flow, 100.0, 5000.0),
                               cfl=0.5))
    return out


def prepare(case, seed):
    s = State()
    s.case = case
    if case["op"] == "batch":
        specs = _specs(case, seed)
        blocks = sum(x.blocks for x in specs)
        s.batch = s.add(sa.Batch(int(blocks * sa.Batch.BYTES_PER_BLOCK * 1.05) + (16 << 20)))
        s.ids = [s.batch.add(x) for x in specs]
        return s
    f = _flow(case)
    walls = case["stretch"]
    s.grid = s.add(sa.CartesianGrid((case["cx"], case["cy"], case["cz"]), (case["bx"], case["by"], case["bz"]),
                                    tuple(zip(f["lo"], f["hi"])), num_exch=NG, periodic=(True, not walls, True),
                                    maps=(None, sa.tanh_map(-1.0, 1.0, TANH_BETA) if walls else None, None)))
    gas = sa.IdealGas(GAMMA, f["R"])
    s.gas, s.flux = gas, _flux(case, gas)
    host = _ghostless(case, _interior(case, seed)).cpu().numpy()
    s.q = s.add(sa.GridArray(s.grid))
    s.exchange = sa.create_exchange(s.q)
    if case["op"] == "host":
        s.host = host
        s.rhs = s.add(sa.GridArray(s.grid, fill=0.0))
        return s
    s.q.upload(host)
    s.exchange.exchange(s.q)
    if walls:
        sa.boundary_fill_wall(s.q, 2, T_WALL)
        sa.boundary_fill_wall(s.q, 3, T_WALL)
    faces = dict(walls=(2, 3), t_wall=T_WALL) if walls else {}
    if case["op"] == "rhs":
        s.rhs = s.add(sa.GridArray(s.grid, fill=0.0))
        if case["increment"]:
            s.rhs.upload(_ghostless(case, _source(case, seed)).cpu().numpy())
    elif case["op"] == "ssprk3":
        s.it = s.add(sa.Integrator(s.q, s.flux, f["dt"], scheme=sa.ssprk3, **faces))
    else:
        s.it = s.add(sa.RKIntegrator(s.q, sa.rk4, f["dt"], gas=gas, flux=s.flux, **faces))
    return s


def run(s):
    case = s.case
    op = case["op"]
    if op == "rhs":
        sa.flux_div(s.q, s.rhs, s.flux, increment=case["increment"])
        return Arrays(s, rhs=s.rhs)
    if op == "host":
        s.q.upload(s.host)
        s.exchange.exchange(s.q)
        if case["stretch"]:
            sa.boundary_fill_wall(s.q, 2, T_WALL)
            sa.boundary_fill_wall(s.q, 3, T_WALL)
        sa.flux_div(s.q, s.rhs, s.flux, increment=False)
        return {"rhs": s.rhs.download()}
    if op == "batch":
        s.batch.step(case["steps"])
        return Ensemble(s)
    s.it.advance(case["steps"])
    out = Arrays(s, q=s.q)
    if case["monitor"]:
        out["wave"] = sa.max_wavespeed(s.q, s.gas)
        out["ke"], out["enstrophy"] = sa.diagnostics(s.q, s.gas)
    return out


class Ensemble(dict):
    """The ensemble's conserved states (one case after the other) and
    histories, read from the engine when looked up."""

    def __init__(self, s):
        super().__init__(state=None, ke=None, enstrophy=None)
        self.s = s

    def __getitem__(self, key):
        b, ids = self.s.batch, self.s.ids
        if key == "state":
            return np.concatenate([b.download(i).reshape(-1) for i in ids])
        return np.concatenate([b.diag(i)[0 if key == "ke" else 1] for i in ids])


# --------------------------------------------------------------------- work ---

def work(case):
    if case["op"] == "batch":
        cells = sum(x.num_cells for x in _specs(case, 0))
        # per step and cell: stage 1 reads and writes 40 B, stages 2 and 3 also read u0
        return {"bytes": 320.0 * cells * case["steps"], "flops": 3.0 * 600.0 * cells * case["steps"]}
    n = _flow(case)["n"]
    cells = float(n[0] * n[1] * n[2])
    flops = FLUXES[case["flux"]]["flops"] * cells
    if case["op"] == "rhs":
        return {"bytes": (120.0 if case["increment"] else 80.0) * cells, "flops": flops}
    if case["op"] == "host":
        stored = case["bx"] * case["by"] * case["bz"] * 40.0
        for c in ("cx", "cy", "cz"):
            stored *= case[c] + 2 * NG
        return {"bytes": 2.0 * stored, "flops": flops}
    stages = 3 if case["op"] == "ssprk3" else 4
    per = 80.0 + 120.0 * (stages - 1)
    return {"bytes": per * cells * case["steps"] + (40.0 * cells if case["monitor"] else 0.0),
            "flops": stages * flops * case["steps"]}


# -------------------------------------------------------------------- exact ---

class _Faces:
    """Views of a padded field around the faces of direction d (0..n along d):
    ``at(v, o)`` is the cell at offset o from the face's right cell (o = -1:
    left cell); a tangential shift moves along another axis."""

    def __init__(self, q, n, d):
        self.q, self.n, self.d = q, n, d

    def at(self, v, o, t=None, s=0):
        a = self.q[v]
        for ax in range(3):
            lo, ln = NG, self.n[ax]
            if ax == self.d:
                lo, ln = NG + o, self.n[ax] + 1
            elif ax == t:
                lo += s
            a = a.narrow(2 - ax, lo, ln)
        return a


def _map_y(f, xi):
    th = torch.tanh(TANH_BETA * xi)
    return TANH_BETA * (1.0 - th * th) / math.tanh(TANH_BETA)


def _face_flux(case, f, F, d):
    """The composed flux (5 fields) on the faces of direction d."""
    R, dx, name, mu0 = f["R"], f["dx"], case["flux"], f["mu"]
    dev = F.q.device
    # d y / d eta at the rows of this direction's faces and cells
    my_face = nl = nr = None
    if case["stretch"]:
        ny = f["n"][1]
        if d == 1:
            my_face = _map_y(f, f["lo"][1] + torch.arange(ny + 1, device=dev, dtype=torch.float64) * dx[1])
        else:
            my_face = _map_y(f, f["lo"][1] + (torch.arange(ny, device=dev, dtype=torch.float64) + 0.5) * dx[1])
        my_face = my_face.view(1, -1, 1)
    # the face normal of a diagonal map has one component, area weighted
    nd = my_face if (case["stretch"] and d != 1) else 1.0

    def cell(o):
        p, t, u, v, w = (F.at(k, o) for k in range(5))
        rho = p / (R * t)
        return p, t, (u, v, w), rho, p / (rho * (GAMMA - 1.0))
    L, Rr = cell(-1), cell(0)

    def gradient(v):
        g = [None] * 3
        for c in range(3):
            if c == d:
                g[c] = (F.at(v, 0) - F.at(v, -1)) / dx[c]
            else:
                g[c] = 0.25 * ((F.at(v, -1, c, 1) - F.at(v, -1, c, -1)) + (F.at(v, 0, c, 1) - F.at(v, 0, c, -1))) / dx[c]
            if c == 1 and my_face is not None:
                g[c] = g[c] / my_face
        return g
    gu = [gradient(U), gradient(V), gradient(W)]        # gu[i][c] = d u_i / d x_c
    gT = gradient(T)
    uf = [0.5 * (L[2][i] + Rr[2][i]) for i in range(3)]
    Tf, pf = 0.5 * (L[1] + Rr[1]), 0.5 * (L[0] + Rr[0])
    div = gu[0][0] + gu[1][1] + gu[2][2]

    # viscous part
    if name in ("keep2_ducros_visc", "weno_visc", "fweno_visc"):
        mu, lam, alpha = mu0, -2.0 * mu0 / 3.0, mu0 / PRANDTL
    else:
        mu = mu0 * Tf ** POWER
        lam, alpha = -0.66666666667 * mu, mu / PRANDTL
    if name == "keep4_wale":
        g2 = [[sum(gu[i][k] * gu[k][j] for k in range(3)) for j in range(3)] for i in range(3)]
        tr = (g2[0][0] + g2[1][1] + g2[2][2]) / 3.0
        ssd = ss = 0.0
        for i in range(3):
            for j in range(3):
                sd = 0.5 * (g2[i][j] + g2[j][i]) - (tr if i == j else 0.0)
                ssd = ssd + sd * sd
                ss = ss + (0.5 * (gu[i][j] + gu[j][i])) ** 2
        rho = pf / (R * Tf)
        mt = rho * (0.5 * 0.06) ** 2 * ssd ** 1.5 / (1e-8 + ss ** 2.5 + ssd ** 1.25)
        mu, lam, alpha = mu + mt, lam - 0.66666666667 * mt, alpha + mt / 0.9
    tau = [mu * (gu[d][b] + gu[b][d]) + (lam * div if b == d else 0.0) for b in range(3)]
    heat = sum(uf[b] * tau[b] for b in range(3)) + (GAMMA * R / (GAMMA - 1.0)) * alpha * gT[d]
    out = [0.0, -nd * heat] + [-nd * tau[b] for b in range(3)]

    # pressure diffusion
    if name in ("keep2_pdiss_visc", "keep2_ducros_visc"):
        if name == "keep2_ducros_visc":
            th = div * div
            cu = [gu[2][1] - gu[1][2], gu[0][2] - gu[2][0], gu[1][0] - gu[0][1]]
            scl = th / (th + sum(c * c for c in cu) + 1e-2)
            eps_p, eps_t = 0.1, 0.05
        else:
            scl, eps_p, eps_t = 0.5, 0.1, 0.1
        irt = 1.0 / (R * Tf)
        k = 0.5 * sum(L[2][i] * Rr[2][i] for i in range(3))
        a = scl * eps_p * (L[0] - Rr[0])
        b = scl * eps_t * (L[1] - Rr[1]) * pf * irt / Tf
        pd = [a * irt - b, a * (k * irt + 1.0 / GAMMA) - 0.5 * k * b] + [(a * irt - b) * uf[i] for i in range(3)]
        out = [o + x for o, x in zip(out, pd)]

    # convective part
    un = lambda c, n: c[2][d] * n        # noqa: E731
    if case["stretch"] and d == 1:
        ncell = {o: 1.0 for o in (-2, -1, 0, 1)}
    else:
        ncell = {o: nd for o in (-2, -1, 0, 1)}
    if name in ("keep2_visc", "keep2_pdiss_visc", "keep2_ducros_visc", "totani_visc"):
        unl, unr = un(L, ncell[-1]), un(Rr, ncell[0])
        c = 0.25 * (L[3] + Rr[3]) * (unl + unr)
        K = sum(L[2][i] * Rr[2][i] for i in range(3))
        conv = [c, 0.5 * c * (L[4] + Rr[4] + K) + 0.5 * (unl * Rr[0] + unr * L[0])]
        for i in range(3):
            m = c * uf[i]
            conv.append(m + nd * pf if i == d else m)
    elif name == "keep4_wale":
        q = [cell(o) for o in (-2, -1, 0, 1)]
        uns = [un(q[i], ncell[i - 2]) for i in range(4)]
        conv = [0.0] * 5
        for ii, a in ((1, 2.0 / 3.0), (2, -1.0 / 12.0)):
            for jj in range(ii):
                x, y = 1 - jj, 1 - jj + ii
                A, B = q[x], q[y]
                c = a * 0.25 * (A[3] + B[3]) * (uns[x] + uns[y])
                conv[0] = conv[0] + 2.0 * c
                conv[1] = conv[1] + c * (sum(A[2][i] * B[2][i] for i in range(3)) + A[4] + B[4]) \
                    + a * (uns[x] * B[0] + uns[y] * A[0])
                for i in range(3):
                    conv[2 + i] = conv[2 + i] + c * (A[2][i] + B[2][i])
                    if i == d:
                        conv[2 + i] = conv[2 + i] + a * (A[0] + B[0]) * nd
    else:
        up, dn = [], []
        for o in (-2, -1, 0, 1):
            p, t, u, rho, e = cell(o)
            k2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
            un_ = u[d] * ncell[o]
            eng = 0.5 * k2 + R * t / (GAMMA - 1.0)
            fl = [rho * un_, rho * un_ * (eng + R * t)] + [rho * un_ * u[i] for i in range(3)]
            fl[2 + d] = fl[2 + d] + p * ncell[o]
            s = torch.sqrt(k2) + torch.sqrt(GAMMA * R * t)
            ds = [rho * s, rho * s * eng] + [rho * s * u[i] for i in range(3)]
            up.append([0.5 * (x + y) for x, y in zip(fl, ds)])
            dn.append([0.5 * (x - y) for x, y in zip(fl, ds)])
        conv = []
        for k in range(5):
            a, b, c = up[0][k], up[1][k], up[2][k]
            x, y, z = dn[1][k], dn[2][k], dn[3][k]
            b0, b1, b2, b3 = (a - b) ** 2 + 1e-16, (b - c) ** 2 + 1e-16, (x - y) ** 2 + 1e-16, (y - z) ** 2 + 1e-16
            # w0 = (1/3)/b0^2 over (1/3)/b0^2 + (2/3)/b1^2
            w0 = b1 * b1 / (b1 * b1 + 2.0 * b0 * b0)
            w3 = b2 * b2 / (b2 * b2 + 2.0 * b3 * b3)
            conv.append(w0 * (1.5 * b - 0.5 * a) + (1.0 - w0) * 0.5 * (b + c)
                        + (1.0 - w3) * 0.5 * (x + y) + w3 * (1.5 * y - 0.5 * z))
    return [a + b for a, b in zip(out, conv)]


def _residual(case, f, q):
    """-div F of the interior field q, (5, nz, ny, nx)."""
    pad = _pad(case, q)
    jac = 1.0
    if case["stretch"]:
        ny = f["n"][1]
        yc = f["lo"][1] + (torch.arange(ny, device=q.device, dtype=torch.float64) + 0.5) * f["dx"][1]
        jac = (1.0 / _map_y(f, yc)).view(1, ny, 1)
    out = torch.zeros_like(q)
    for d in range(3):
        flux = _face_flux(case, f, _Faces(pad, f["n"], d), d)
        ax = 2 - d
        for v in range(5):
            if not torch.is_tensor(flux[v]):
                continue
            n = f["n"][d]
            out[v] -= (flux[v].narrow(ax, 1, n) - flux[v].narrow(ax, 0, n)) * jac / f["dx"][d]
    return out


def _cons(q, R):
    rho = q[P] / (R * q[T])
    return torch.stack([rho, 0.5 * rho * (q[U] ** 2 + q[V] ** 2 + q[W] ** 2) + q[P] / (GAMMA - 1.0),
                        rho * q[U], rho * q[V], rho * q[W]])


def _prim(c, R):
    u = c[2:] / c[0]
    p = (GAMMA - 1.0) * (c[1] - 0.5 * c[0] * (u * u).sum(0))
    return torch.stack([p, p / (R * c[0]), u[0], u[1], u[2]])


def _steps(case, f, q, dt, steps, table):
    """steps of an explicit table (rows a, weights b) in conserved variables."""
    a, b = table
    for _ in range(steps):
        u0, k = _cons(q, f["R"]), []
        for row in a:
            u = u0.clone()
            for c, r in zip(row, k):
                if c:
                    u += (dt * c) * r
            k.append(_residual(case, f, _prim(u, f["R"])))
        for c, r in zip(b, k):
            u0 += (dt * c) * r
        q = _prim(u0, f["R"])
    return q


SSPRK3 = (((), (1.0,), (0.25, 0.25)), (1.0 / 6.0, 1.0 / 6.0, 2.0 / 3.0))
RK4 = (((), (0.5,), (0.0, 0.5), (0.0, 0.0, 1.0)), (1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0))


def _diagnose(case, f, q, R):
    """Volume-averaged kinetic energy and enstrophy (second-order central
    differences in computational coordinates) of the interior field q."""
    pad, n = _pad(case, q), f["n"]

    def d(v, ax):
        def s(o):
            a = pad[v]
            for k in range(3):
                a = a.narrow(2 - k, NG + (o if k == ax else 0), n[k])
            return a
        return 0.5 * (s(1) - s(-1)) / f["dx"][ax]
    om = (d(W, 1) - d(V, 2), d(U, 2) - d(W, 0), d(V, 0) - d(U, 1))
    ke = 0.5 * (q[P] / (R * q[T])) * (q[U] ** 2 + q[V] ** 2 + q[W] ** 2)
    return float(ke.mean()), float(0.5 * sum(o * o for o in om).mean())


def _exact_ensemble(case, seed):
    dev = _device()
    states, kes, ens = [], [], []
    for s in _specs(case, seed):
        nx, ny, nz = s.cells
        tgv = s.kind == "tgv"
        length = 2.0 * math.pi if tgv else 10.0
        dx = [length / c for c in s.cells]
        x, y, z = ((torch.arange(s.cells[a], device=dev, dtype=torch.float64) + 0.5) * dx[a] for a in range(3))
        x, y, z = x.view(1, 1, nx), y.view(1, ny, 1), z.view(nz, 1, 1)
        one = torch.ones((nz, ny, nx), device=dev, dtype=torch.float64)
        if tgv:
            R = 1.0 / (s.mach * s.mach * GAMMA)
            mu = 1.0 / s.reynolds
            p = R + (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0
            u, v = torch.sin(x) * torch.cos(y) * torch.cos(z), -torch.cos(x) * torch.sin(y) * torch.cos(z)
            q = torch.stack([p * one, one, u * one, v * one, 0.0 * one])
            speed = 1.0 + math.sqrt(GAMMA * (R + 0.75))
        else:
            R, beta = 1.0 / GAMMA, 5.0 * s.mach
            mu = s.mach / s.reynolds
            xr, yr = x - 5.0, y - 5.0
            r2 = xr * xr + yr * yr
            e = torch.exp(0.5 * (1.0 - r2)) * beta / (2.0 * math.pi)
            t = 1.0 - (GAMMA - 1.0) * beta * beta / (8.0 * math.pi ** 2) * torch.exp(1.0 - r2)
            p = t ** (1.0 / (GAMMA - 1.0)) * R * t
            q = torch.stack([p * one, t * one, (s.mach - yr * e) * one, xr * e * one, 0.0 * one])
            speed = s.mach + beta / (2.0 * math.pi) + 1.0
        c = dict(flux="keep2_visc", stretch=False)
        f = dict(R=R, mu=mu, dx=dx, n=s.cells)
        for _ in range(case["steps"]):
            ke, en = _diagnose(c, f, q, R)
            kes.append(ke)
            ens.append(en)
            q = _steps(c, f, q, s.cfl * min(dx) / speed, 1, SSPRK3)
        u = _cons(q, R).reshape(5, nz // 16, 16, ny // 16, 16, nx // 16, 16)
        states.append(u.permute(1, 3, 5, 0, 2, 4, 6).reshape(-1).cpu())
    return {"state": torch.cat(states).numpy(), "ke": np.array(kes), "enstrophy": np.array(ens)}


def exact(case, seed):
    if case["op"] == "batch":
        return _exact_ensemble(case, seed)
    f, q = _flow(case), _interior(case, seed)
    if case["op"] in ("rhs", "host"):
        r = _residual(case, f, q)
        if case["increment"]:
            r += _source(case, seed)
        return {"rhs": _ghostless(case, r).cpu().numpy()}
    q = _steps(case, f, q, f["dt"], case["steps"], SSPRK3 if case["op"] == "ssprk3" else RK4)
    out = {"q": _to_blocks(case, _pad(case, q)).cpu().numpy()}
    if case["monitor"]:
        speed = torch.sqrt(GAMMA * f["R"] * q[T]) + torch.sqrt(q[U] ** 2 + q[V] ** 2 + q[W] ** 2)
        out["wave"] = float(speed.max())
        out["ke"], out["enstrophy"] = _diagnose(case, f, q, f["R"])
    return out
