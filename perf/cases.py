"""The work that users of this framework have it do, as cases that can be timed.

Every case steps simulations (or differentiates through them) by the public
entry points of picongpu_amd, over the range of sizes, shapes, pushers,
solvers and boundaries the setups, tests and bench.py use:

- "box": a periodic plasma box, one or two species, advanced by `steps` full
  steps: eagerly ("step"), replayed from the captured graphs ("graph") or by
  the stage calls of a host code that keeps its own step loop ("stages");
- "laser": the laser-plasma geometry with open borders;
- "ensemble": independent boxes advanced by batched launches;
- "adjoint": the differentiable form, forward and backward.

A pass advances the state it is given, as a simulation does, and ends where a
program would look at the fields: E and B are read into the program's own
pinned buffers. They hold the effect of every particle's move (its current is
in E); the particles stay in the context, as between a simulation's outputs.
"""
import ctypes
import dataclasses
import math

import numpy as np
import torch

from picongpu_amd import abi, adjoint, setups

C_SI = 2.99792458e8
ME_SI = 9.1093837139e-31
QE_SI = 1.602176634e-19
EPS0_SI = 8.8541878188e-12

# largest particle count that is loaded from arrays (larger boxes are filled on the device)
MAX_LOADED = 2_200_000


def _box(name, grid, ppc, shape, steps, **more):
    case = {"name": name, "kind": "box", "nx": grid[0], "ny": grid[1], "nz": grid[2], "ppc": ppc, "shape": shape,
            "steps": steps, "species": 1, "drift": 0.0, "pusher": abi.PUSHER_BORIS, "solver": abi.SOLVER_YEE,
            "call": "step", "loaded": True, "emz": False, "binomial": False, "quiet": False, "monitor": False}
    case.update(more)
    return case


def _laser(name, grid, steps, laser, absorber, call):
    return {"name": name, "kind": "laser", "nx": grid[0], "ny": grid[1], "nz": grid[2], "ppc": 4, "steps": steps,
            "laser": laser, "absorber": absorber, "call": call}


def listed():
    return [
        # the smallest simulations: unit checks and parameter scans of a few
        # thousand particles, where a step is launches and latency
        _box("tiny_tsc", (16, 16, 12), 4, 2, 10),
        # the plain thermal box, replayed from graphs as a production loop runs it
        _box("thermal_64_cic", (64, 64, 64), 8, 1, 20, call="graph"),
        # counter-streaming beams on a ragged grid (rings that do not divide evenly)
        _box("streams_72x88x36_tsc", (72, 88, 36), 9, 2, 10, drift=0.25),
        # monitored run: steps with the field energies and the Gauss residual after them
        _box("monitor_48x40x44_pqs", (48, 40, 44), 6, 3, 10, monitor=True),
        # the shear-flow growth-rate test: thin in z, quiet start, 25 + 25 particles per cell
        _box("khi_192x512x12_tsc", (192, 512, 12), 25, 2, 5, species=2, loaded=False, quiet=True),
        # the two-species shear flow at full size, the framework's benchmark
        _box("shear_256_tsc", (256, 256, 256), 16, 2, 5, species=2, drift=0.2, loaded=False),
        # a host code's own step loop over the stage calls, unfused deposit
        _box("stages_96x64x64_tsc_emz", (96, 64, 64), 8, 2, 5, species=2, drift=0.1, loaded=False, call="stages",
             pusher=abi.PUSHER_HIGUERA_CARY, emz=True, binomial=True),
        # laser wakefield at full size: PQS, Vay, Lehe, PML with its weight damping
        _laser("laser_192x1536x192", (192, 1536, 192), 5, "initial", "pml", "step"),
        # a small wakefield scan point: injected pulse, exponential absorber, graphs
        _laser("laser_96x512x64_injected", (96, 512, 64), 10, "incident", "exponential", "graph"),
        # batched parameter scan
        {"name": "ensemble_32", "kind": "ensemble", "members": 32, "lo": 32, "hi": 96, "ppc_lo": 2, "ppc_hi": 16,
         "steps": 5},
        # gradients of a probe's field energy: a small fit and the full-size box
        {"name": "adjoint_16", "kind": "adjoint", "nx": 16, "ny": 16, "nz": 16, "ppc": 2, "steps": 12, "every": 5},
        {"name": "adjoint_64", "kind": "adjoint", "nx": 64, "ny": 64, "nz": 64, "ppc": 8, "steps": 40, "every": 20},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """Cells per axis, multiples of the supercell's 8 x 8 x 4."""
    return tuple(max(step * 2, step * (_loguniform(rng, lo, hi) // step)) for step in (8, 8, 4))


def draw(rng):
    kind = rng.choice(["box", "box", "box", "laser", "ensemble", "adjoint"])
    if kind == "laser":
        grid = (8 * rng.randint(7, 20), 8 * rng.randint(40, 96), 4 * rng.randint(14, 40))
        case = _laser("", grid, rng.randint(4, 10), rng.choice(["initial", "incident"]),
                      rng.choice(["pml", "pml", "exponential"]), rng.choice(["step", "graph"]))
    elif kind == "ensemble":
        case = {"name": "", "kind": "ensemble", "members": _loguniform(rng, 3, 24), "lo": 32,
                "hi": rng.choice([48, 64, 96]), "ppc_lo": 2, "ppc_hi": rng.choice([4, 8, 16]),
                "steps": rng.randint(3, 8)}
    elif kind == "adjoint":
        g = _grid(rng, 16, 64)
        ppc = _loguniform(rng, 2, 8)
        case = {"name": "", "kind": "adjoint", "nx": g[0], "ny": g[1], "nz": g[2], "ppc": ppc,
                "steps": rng.randint(8, 40), "every": rng.randint(4, 20)}
    else:
        ppc = _loguniform(rng, 2, 32)
        species = rng.choice([1, 1, 2])
        while True:
            g = _grid(rng, 16, 192)
            n = g[0] * g[1] * g[2] * ppc * species
            if n <= 60_000_000:
                break
        loaded = species == 1 and n <= MAX_LOADED
        case = _box("", g, ppc, rng.choice([1, 2, 3]), rng.randint(5, 12), species=species,
                    drift=rng.choice([0.0, 0.1, 0.25]), loaded=loaded, call=rng.choice(["step", "graph", "stages"]),
                    monitor=rng.random() < 0.2)
        if rng.random() < 0.4:
            case.update(pusher=rng.choice([abi.PUSHER_BORIS, abi.PUSHER_VAY, abi.PUSHER_HIGUERA_CARY]),
                        solver=rng.choice([abi.SOLVER_YEE, abi.SOLVER_LEHE]), emz=rng.random() < 0.3,
                        binomial=rng.random() < 0.3)
    del case["name"]
    return case


# -- what a program has in hand before the call --------------------------------

def _box_setup(case, seed):
    grid = (case["nx"], case["ny"], case["nz"])
    if case["quiet"]:
        st = setups.khi_growth_rate(grid=grid, seed=2 * seed)
        if case["ppc"] != st.typical_ppc:
            raise ValueError("the quiet start has 25 particles per cell")
    elif case["species"] == 2:
        st = setups.kelvin_helmholtz(grid=grid, ppc=case["ppc"], shape=case["shape"], seed=2 * seed)
        ud = (setups.gamma_beta(case["drift"]), 0.0, 0.0)
        st.species = [dataclasses.replace(s, u_drift=ud) for s in st.species]
        st.b_noise_seed = seed + 1
    elif case["drift"]:
        st = setups.two_stream(grid=grid, ppc=case["ppc"], beta=case["drift"], seed=seed)
    else:
        st = setups.thermal(grid=grid, ppc=case["ppc"], seed=seed)
    solver = abi.CURRENT_SOLVER_EMZ if case["emz"] else abi.CURRENT_SOLVER_ESIRKEPOV
    st.species = [dataclasses.replace(s, shape=case["shape"], pusher=case["pusher"], current_solver=solver)
                  for s in st.species]
    st.solver = case["solver"]
    st.current_interpolation = abi.CURRENT_BINOMIAL if case["binomial"] else abi.CURRENT_NONE
    return st


def _arrays(case, setup, seed):
    """Seeded particles of a one-species box on the GPU: the k-th particle of
    every cell after the (k-1)-th, as the device's own start places them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    nx, ny, nz = setup.grid
    s = setup.species[0]
    cells = nx * ny * nz
    i = torch.arange(cells, device="cuda")
    cell = torch.stack([i % nx, (i // nx) % ny, i // (nx * ny)], dim=1).to(torch.int32).repeat(s.ppc, 1)
    n = cells * s.ppc
    pos = torch.rand((n, 3), generator=gen, device="cuda")
    u = torch.randn((n, 3), generator=gen, device="cuda") * torch.tensor(s.u_th, device="cuda")
    sign = 1.0 - 2.0 * (torch.arange(s.ppc, device="cuda") % 2).repeat_interleave(cells)
    u = u + sign[:, None] * torch.tensor(s.u_drift, device="cuda")
    weight = np.float32(s.density_si * math.prod(setup.cell_si) / s.ppc)
    typical = setup.density_si * math.prod(setup.cell_si) / setup.typical_ppc
    mom = u * float(weight / typical)
    return cell, pos, mom, torch.full((n,), float(weight), device="cuda")


def _field_buffers(ncells):
    return [torch.empty((3, ncells), dtype=torch.float32, pin_memory=True) for _ in range(2)]


def _read_fields(sim, buffers):
    for field, buf in zip((abi.FIELD_E, abi.FIELD_B), buffers):
        out = ctypes.cast(buf.data_ptr(), ctypes.POINTER(ctypes.c_float))
        abi.check(sim.lib.pic_read_field(sim.h, field, out), "pic_read_field")


def _prepare_sim(case, seed):
    if case["kind"] == "laser":
        grid = (case["nx"], case["ny"], case["nz"])
        setup = setups.laser_plasma(grid=grid, ppc=case["ppc"], seed=2 * seed, laser=case["laser"],
                                    absorber=case["absorber"])
    else:
        setup = _box_setup(case, seed)
    sim = abi.Simulation(setup.config())
    if case["kind"] == "box" and case["loaded"]:
        cell, pos, mom, w = (t.cpu().numpy() for t in _arrays(case, setup, seed))
        sim.load_particles(0, cell, pos, mom, w)
    else:
        setups.init_device(sim, setup)
    if case["kind"] == "laser" and case["laser"] == "incident":
        # the pulse's centre passes the Huygens surface some hundred steps after the start
        sim.set_step(400 + seed % 64)
    return {"case": case, "sim": sim, "fields": _field_buffers(setup.ncells)}


def _prepare_ensemble(case, seed):
    # the members' sizes come with the case, their particles from the seed
    sts = setups.ensemble(n=case["members"], lo=case["lo"], hi=case["hi"],
                          ppc_range=(case["ppc_lo"], case["ppc_hi"]))
    ens = abi.Ensemble([st.config() for st in sts])
    for i, (member, st) in enumerate(zip(ens.members, sts)):
        st.species = [dataclasses.replace(s, seed=seed * 1000 + i) for s in st.species]
        setups.init_device(member, st)
    return {"case": case, "ensemble": ens, "fields": [_field_buffers(st.ncells) for st in sts]}


def _pulse(grid, seed):
    """A Gaussian pulse along x with seeded amplitude and phase, E_y and B_z in
    PIC units of a field, on the Yee positions."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    a, phase = (torch.rand(2, generator=gen, device="cuda", dtype=torch.float64) + 0.5).tolist()
    nx, ny, nz = grid
    x, y, z = (torch.arange(n, device="cuda", dtype=torch.float64) - n / 2 for n in (nx, ny, nz))

    def at(dx, dy, dz):
        xs, ys, zs = (x + dx)[None, None, :], (y + dy)[None, :, None], (z + dz)[:, None, None]
        env = torch.exp(-((xs / (0.2 * nx)) ** 2) - (ys / (0.25 * ny)) ** 2 - (zs / (0.25 * nz)) ** 2)
        return (a * env * torch.cos(2 * math.pi * xs / 8.0 + phase)).reshape(-1)

    zero = torch.zeros(nx * ny * nz, device="cuda", dtype=torch.float64)
    return torch.stack([zero, at(0.0, 0.5, 0.0), zero]), torch.stack([zero, zero, at(0.5, 0.5, 0.0)])


def _adjoint_setup(case, seed):
    return setups.differentiable(grid=(case["nx"], case["ny"], case["nz"]), ppc=case["ppc"], seed=seed)


def _adjoint_inputs(case, seed):
    """Initial fields (an a0 of 0.5 to 1.5) and the particles of a cold plasma
    in tiles of 8 x 4 x 1 cells, slot by slot inside a tile."""
    setup = _adjoint_setup(case, seed)
    unit = adjoint_unit(setup)
    e0, b0 = (f * unit for f in _pulse(setup.grid, seed))
    nx, ny, nz = setup.grid
    gen = torch.Generator(device="cuda").manual_seed(seed)
    tiles = torch.arange(nx // 8 * (ny // 4) * nz, device="cuda")
    loc = torch.arange(32, device="cuda")
    shape = (tiles.numel(), case["ppc"], 32)
    gx = ((tiles % (nx // 8)) * 8)[:, None, None] + (loc % 8)[None, None, :]
    gy = (((tiles // (nx // 8)) % (ny // 4)) * 4)[:, None, None] + (loc // 8)[None, None, :]
    gz = (tiles // (nx // 8 * (ny // 4)))[:, None, None] + 0 * loc[None, None, :]
    cell = torch.stack([g.expand(shape).reshape(-1) for g in (gx, gy, gz)]).to(torch.int32)
    pos = torch.rand(cell.shape, generator=gen, device="cuda")
    weight = float(np.float32(setup.density_si * math.prod(setup.cell_si) / case["ppc"]))
    w = torch.full((cell.shape[1],), weight, device="cuda")
    return setup, e0.float().double(), b0.float().double(), cell, pos, torch.zeros_like(pos), w


def _prepare_adjoint(case, seed):
    setup, e0, b0, cell, pos, mom, w = _adjoint_inputs(case, seed)
    pic = adjoint.DifferentiablePIC(setup, *(t.cpu().numpy() for t in (cell, pos, mom, w)), nsteps=case["steps"],
                                    checkpoint_every=case["every"])
    return {"case": case, "pic": pic, "e0": e0.requires_grad_(), "b0": b0.requires_grad_()}


def prepare(case, seed):
    if case["kind"] == "ensemble":
        return _prepare_ensemble(case, seed)
    if case["kind"] == "adjoint":
        return _prepare_adjoint(case, seed)
    return _prepare_sim(case, seed)


# -- one pass -------------------------------------------------------------------

def _probe_energy(grid, e, b):
    """Field energy in the middle of the box (half of every axis)."""
    nx, ny, nz = grid
    total = 0.0
    for f in (e, b):
        probe = f.reshape(3, nz, ny, nx)[:, nz // 4:nz - nz // 4, ny // 4:ny - ny // 4, nx // 4:nx - nx // 4]
        total = total + 0.5 * (probe * probe).sum()
    return total


def _run_adjoint(state):
    pic, e0, b0 = state["pic"], state["e0"], state["b0"]
    e, b = pic.fields(e0, b0)
    ge, gb = torch.autograd.grad(_probe_energy(pic.setup.grid, e, b), (e0, b0))
    return {"E": e.detach(), "B": b.detach(), "dE0": ge, "dB0": gb}


def _stages(sim):
    sim.current_reset()
    sim.push(-1, fuse_deposit=False)
    sim.shift()
    sim.update_before_current()
    sim.deposit()
    sim.add_current()
    sim.update_after_current()


def run(state):
    case = state["case"]
    if case["kind"] == "adjoint":
        return _run_adjoint(state)
    if case["kind"] == "ensemble":
        state["ensemble"].step_graph(case["steps"])
        for member, buffers in zip(state["ensemble"].members, state["fields"]):
            _read_fields(member, buffers)
        return {"E": [b[0] for b in state["fields"]], "B": [b[1] for b in state["fields"]]}
    sim = state["sim"]
    if case["call"] == "stages":
        for _ in range(case["steps"]):
            _stages(sim)
    elif case["call"] == "graph":
        sim.step_graph(case["steps"])
    else:
        sim.step(case["steps"])
    out = {}
    if case.get("monitor"):
        out["energy"] = sim.field_energy()
        out["gauss"] = sim.gauss_residual()
    _read_fields(sim, state["fields"])
    out["E"], out["B"] = state["fields"]
    return out


# -- what a pass cannot do without -----------------------------------------------

def _particle_flops(support):
    """Gather of six components, push, move and Esirkepov deposit."""
    s = support
    gather = 6 * (2 * (s ** 3 + s ** 2 + s) + 8 * s)
    deposit = 3 * (9 * s * s + 4 * s * s * (s - 1)) + 30 * s
    return gather + 160 + deposit


def work(case):
    """Bytes: per step and particle the 31 B of its attributes read and 24 B
    of position and momentum written, per step and cell E, B and J once for
    the particles (36 B) and once for the field update (60 B), and the fields
    read out. The backward pass of the differentiable form recomputes the
    forward and carries 48 B of FP64 adjoints per particle and 48 B per cell."""
    if case["kind"] == "adjoint":
        cells = case["nx"] * case["ny"] * case["nz"]
        n = cells * case["ppc"]
        step = n * 55 + cells * 96
        back = n * (31 + 2 * 48) + cells * (24 + 2 * 48 + 24)
        return {"bytes": float(case["steps"] * (2 * step + back) + 4 * 24 * cells),
                "flops": float(case["steps"] * (n * 4 * _particle_flops(2) + cells * 200))}
    if case["kind"] == "ensemble":
        sts = setups.ensemble(n=case["members"], lo=case["lo"], hi=case["hi"],
                              ppc_range=(case["ppc_lo"], case["ppc_hi"]))
        cells = sum(st.ncells for st in sts)
        n, support = sum(st.mobile_particles() for st in sts), 3
    elif case["kind"] == "laser":
        cells = case["nx"] * case["ny"] * case["nz"]
        behind = max(0, case["ny"] - 400)  # the ramp starts 400 cells from the border
        n, support = case["nx"] * behind * case["nz"] * case["ppc"], 4
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
        n, support = cells * case["ppc"] * case["species"], case["shape"] + 1
    return {"bytes": float(case["steps"] * (n * 55 + cells * 96) + 24 * cells),
            "flops": float(case["steps"] * (n * _particle_flops(support) + cells * 60))}


# -- the same in 64 bits ------------------------------------------------------------

def _units(setup):
    """Length, charge and field constants in PIC units (dt = c = 1, the mass and
    charge of a typical macro-particle)."""
    typical = setup.density_si * math.prod(setup.cell_si) / setup.typical_ppc
    length, mass, charge = C_SI * setup.dt_si, ME_SI * typical, QE_SI * typical
    eps0 = EPS0_SI * mass * length ** 3 / (setup.dt_si ** 2 * charge ** 2)
    return [c / length for c in setup.cell_si], 1.0 / typical, eps0, mass * length / (setup.dt_si ** 2 * charge)


def adjoint_unit(setup):
    """Field of a0 = 1 at 0.8 um in PIC units."""
    return ME_SI * C_SI * (2 * math.pi * C_SI / 0.8e-6) / QE_SI / _units(setup)[3]


def _assign(support, x):
    """The assignment function of the shape at a distance of x cells."""
    a = x.abs()
    zero = torch.zeros_like(a)
    if support == 2:
        return torch.where(a < 1, 1 - a, zero)
    if support == 3:
        return torch.where(a < 0.5, 0.75 - a * a, torch.where(a < 1.5, 0.5 * (1.5 - a) ** 2, zero))
    return torch.where(a < 1, (4 - 6 * a ** 2 + 3 * a ** 3) / 6, torch.where(a < 2, (2 - a) ** 3 / 6, zero))


def _nodes(base, count, n, x, support, offset):
    """Wrapped node indices of one axis (particles x count) and their weights."""
    node = base[:, None] + torch.arange(count, device=x.device)
    return node % n, _assign(support, node + offset - x[:, None])


def _flat(ix, iy, iz, grid):
    return ix[:, None, None, :] + grid[0] * (iy[:, None, :, None] + grid[1] * iz[:, :, None, None])


def _outer(wx, wy, wz):
    return wx[:, None, None, :] * wy[:, None, :, None] * wz[:, :, None, None]


def _gather(field, component, x, grid, support, electric):
    axes = []
    for d in range(3):
        offset = 0.5 * ((d == component) == electric)
        at = x[d].detach() - offset
        base = torch.floor(at + (0.5 if support == 3 else 0.0)).long() - (support - 1) // 2
        axes.append(_nodes(base, support, grid[d], x[d], support, offset))
    index = _flat(*(a[0] for a in axes), grid)
    value = field[component].index_select(0, index.reshape(-1)).reshape(index.shape)
    return (value * _outer(*(a[1] for a in axes))).sum(dim=(1, 2, 3))


def _current(x0, x1, charge, grid, cell, support):
    """Esirkepov's current of the moves x0 -> x1 (cells)."""
    half = 0.5 if support == 3 else 0.0
    index, s0, ds = [], [], []
    for d in range(3):
        lower = torch.minimum(torch.floor(x0[d].detach() + half), torch.floor(x1[d].detach() + half)).long()
        base = lower - (support - 1) // 2
        node, a = _nodes(base, support + 1, grid[d], x0[d], support, 0.0)
        index.append(node)
        s0.append(a)
        ds.append(_nodes(base, support + 1, grid[d], x1[d], support, 0.0)[1] - a)
    flat = _flat(*index, grid).reshape(-1)
    volume = cell[0] * cell[1] * cell[2]
    out = []
    for c in range(3):
        a, b = (c + 1) % 3, (c + 2) % 3
        along = -torch.cumsum(ds[c], dim=1) * (charge * cell[c] / volume)[:, None]

        def spread(va, vb):
            w = [None, None, None]
            w[a], w[b], w[c] = va, vb, along
            return _outer(*w)

        j = spread(s0[a] + 0.5 * ds[a], s0[b]) + spread(0.5 * s0[a] + ds[a] / 3, ds[b])
        out.append(torch.zeros(math.prod(grid), dtype=torch.float64, device=flat.device)
                   .index_add(0, flat, j.reshape(-1)))
    return torch.stack(out)


def _curl(f, grid, cell, sign):
    """curl with forward (sign 1) or backward (sign -1) differences."""
    g = f.reshape(3, grid[2], grid[1], grid[0])

    def der(c, d):
        return sign * (torch.roll(g[c], -sign, dims=2 - d) - g[c]) / cell[d]

    return torch.stack([der(2, 1) - der(1, 2), der(0, 2) - der(2, 0), der(1, 0) - der(0, 1)]).reshape(3, -1)


def _step(e, b, x, p, mass, charge, grid, cell, eps0, support):
    """One step: gather, Boris, move, Esirkepov, Yee. x: (3, n) in cells."""
    ef = torch.stack([_gather(e, c, x, grid, support, True) for c in range(3)])
    bf = torch.stack([_gather(b, c, x, grid, support, False) for c in range(3)])
    minus = p + 0.5 * charge * ef
    gamma = torch.sqrt(1 + (minus * minus).sum(0) / mass ** 2)
    t = 0.5 * charge / mass * bf / gamma
    s = 2 * t / (1 + (t * t).sum(0))
    prime = minus + torch.linalg.cross(minus, t, dim=0)
    p = minus + torch.linalg.cross(prime, s, dim=0) + 0.5 * charge * ef
    v = p / torch.sqrt(mass ** 2 + (p * p).sum(0))
    x1 = x + v / torch.tensor(cell, dtype=torch.float64, device=x.device)[:, None]
    j = _current(x, x1, charge, grid, cell, support)
    b = b - 0.5 * _curl(e, grid, cell, 1)
    e = e + _curl(b, grid, cell, -1) - j / eps0
    b = b - 0.5 * _curl(e, grid, cell, 1)
    n = torch.tensor(grid, dtype=torch.float64, device=x.device)[:, None]
    return e, b, x1 - n * torch.floor(x1.detach() / n), p


def _exact_box(case, seed):
    setup = _box_setup(case, seed)
    cell, per_weight, eps0, _ = _units(setup)
    at, pos, mom, w = _arrays(case, setup, seed)
    x, p = (at + pos.double()).T.contiguous(), mom.double().T.contiguous()
    mass, charge = w.double() * per_weight, -w.double() * per_weight
    e = torch.zeros((3, setup.ncells), dtype=torch.float64, device="cuda")
    b = e.clone()
    for _ in range(case["steps"]):
        e, b, x, p = _step(e, b, x, p, mass, charge, setup.grid, cell, eps0, case["shape"] + 1)
    out = {"E": e.cpu(), "B": b.cpu()}
    if case["monitor"]:
        out.update(energy=None, gauss=None)
    return out


def _exact_adjoint(case, seed):
    setup, e0, b0, at, pos, mom, w = _adjoint_inputs(case, seed)
    cell, per_weight, eps0, _ = _units(setup)
    mass, charge = w.double() * per_weight, -w.double() * per_weight

    def step(e, b, x, p):
        return _step(e, b, x, p, mass, charge, setup.grid, cell, eps0, 2)

    e0.requires_grad_()
    b0.requires_grad_()
    # the states of every step, then one step's graph at a time backwards
    states = [(e0, b0, at + pos.double(), mom.double())]
    with torch.no_grad():
        for _ in range(case["steps"]):
            states.append(step(*states[-1]))
    e, b = (f.detach().requires_grad_() for f in states[-1][:2])
    grads = torch.autograd.grad(_probe_energy(setup.grid, e, b), (e, b)) + (torch.zeros_like(states[0][2]),) * 2
    for state in reversed(states[:-1]):
        inputs = [t.detach().requires_grad_() for t in state]
        grads = torch.autograd.grad(step(*inputs), inputs, grads)
    return {"E": e.detach(), "B": b.detach(), "dE0": grads[0], "dB0": grads[1]}


def exact(case, seed):
    """For boxes loaded from arrays with the Boris pusher, Esirkepov's current
    and the Yee solver, and for the differentiable form. The others start on
    the device from the framework's own generator, or are too large."""
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    plain = (case["kind"] == "box" and case["loaded"] and case["pusher"] == abi.PUSHER_BORIS and not case["emz"]
             and case["solver"] == abi.SOLVER_YEE and not case["binomial"])
    return _exact_box(case, seed) if plain else None
