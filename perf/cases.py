"""The work whose speed is followed: what programs have this package do, through its public calls.

``listed()`` names the cases, ``draw`` makes more of the same ranges, ``prepare`` builds what a
program holds before the call (inputs from a seed; a model, a list or a simulation), ``run`` is
one pass, ``work`` what that pass cannot do without and ``exact`` its results in 64 bits by
plain torch. A case is a dict of plain values; its ``path`` says which calls it makes:

- ``md``: ``md.nvt`` / ``md.npt``, ``run`` for some steps, then ``state`` (a production run);
- ``md_batch``: many simulations stepped together, a ``SimulationBatch`` per kind of potential
  on a stream of its own (a server's resident short runs);
- ``evaluate``: one frame from positions alone: a new ``NeighborList``, E, F and W;
- ``follow``: a kept list over consecutive frames, ``update`` and E, F, W at each (a program
  with an integrator of its own);
- ``differentiate``: E, F, W and parameter gradients of a user's energy around a model;
- ``batch``: E, F and W of many systems of uneven size, new frames each pass;
- ``fit``: ``training.fit`` on labeled frames, from the labels to the trained parameters.
"""

import math
import random

import numpy as np
import torch

from nabladyn_amd import md, potential, quantity, training, units, workloads
from nabladyn_amd.batch import Batch
from nabladyn_amd.neighbors import NeighborList

_KT = units.BOLTZMANN * 120.0
_TAU, _TIMESTEP, _SPACING = 0.1, 0.004, 0.016  # ps


def listed():
    return [
        # the smallest simulation: a few hundred atoms, set by launches and their gaps
        {"name": "md_nvt_argon_512", "path": "md", "ensemble": "nvt", "atoms": 512,
         "potential": "lj", "dtype": "float32", "skin": 0.1, "steps": 100, "ry": 1.0, "rz": 1.0},
        # an everyday liquid box at the default skin
        {"name": "md_nvt_argon_32768", "path": "md", "ensemble": "nvt", "atoms": 32768,
         "potential": "lj", "dtype": "float32", "skin": 0.1, "steps": 100, "ry": 1.0, "rz": 1.0},
        # the benchmark's system, the largest simulation
        {"name": "md_nvt_argon_2097152", "path": "md", "ensemble": "nvt", "atoms": 2097152,
         "potential": "lj", "dtype": "float32", "skin": 0.2, "steps": 50, "ry": 1.0, "rz": 1.0},
        # constant pressure, two types, double precision, an odd count in an uneven box
        {"name": "md_npt_mixture_10007_f64", "path": "md", "ensemble": "npt", "atoms": 10007,
         "potential": "mixture", "dtype": "float64", "skin": 0.1, "steps": 50, "ry": 1.1,
         "rz": 1.3},
        # a server's resident runs: 14 systems of 320 to 196,608 atoms, LJ and tables
        {"name": "md_batch_14_systems", "path": "md_batch", "systems": 14, "low": 320,
         "high": 196608, "dtype": "float32", "skin": 0.2, "steps": 50},
        # one small frame evaluated: host work and launches count
        {"name": "evaluate_lj_864", "path": "evaluate", "atoms": 864, "potential": "lj",
         "dtype": "float32", "order": "lattice", "ry": 1.0, "rz": 1.0},
        # one large frame of a table, its atoms in a file's order rather than a spatial one
        {"name": "evaluate_table_205875_shuffled", "path": "evaluate", "atoms": 205875,
         "potential": "table", "dtype": "float32", "order": "shuffled", "ry": 1.4, "rz": 1.7},
        # a program's own integrator at full size, the list reused or rebuilt as atoms move
        {"name": "follow_lj_2097152", "path": "follow", "atoms": 2097152, "potential": "lj",
         "dtype": "float32", "order": "lattice", "skin": 0.1, "frames": 6, "ry": 1.0, "rz": 1.0},
        # the same with a sum of two models over an inner and an outer list, in double precision
        {"name": "follow_sum_50653_f64", "path": "follow", "atoms": 50653, "potential": "sum",
         "dtype": "float64", "order": "shuffled", "skin": 0.1, "frames": 6, "ry": 1.0,
         "rz": 1.0},
        # a user's energy: a two-type model plus a restraint, and its parameter gradients
        {"name": "differentiate_mixture_32768", "path": "differentiate", "atoms": 32768,
         "potential": "mixture", "dtype": "float32", "order": "lattice", "ry": 1.0, "rz": 1.0},
        # 256 independent systems of 64 to 32,768 atoms, half LJ and half tables
        {"name": "batch_256_systems", "path": "batch", "systems": 256, "low": 64, "high": 32768,
         "dtype": "float32"},
        # force matching of a 200-knot table on 64 coarse-grained frames
        {"name": "fit_table_64x4096", "path": "fit", "frames": 64, "atoms": 4096, "batch": 64,
         "updates": 50, "potential": "table", "dtype": "float32"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(("md", "md", "md_batch", "evaluate", "evaluate", "follow", "follow",
                       "differentiate", "batch", "fit"))
    case = {"path": path, "dtype": rng.choice(("float32", "float32", "float32", "float64"))}
    box = {"ry": round(rng.uniform(1, 2), 3), "rz": round(rng.uniform(1, 2), 3)}
    order = rng.choice(("lattice", "shuffled"))
    small = case["dtype"] == "float64"
    if path == "md":
        ensemble, kind = rng.choice((("nvt", "lj"), ("nvt", "table"), ("nvt", "mixture"),
                                     ("nvt", "sum"), ("npt", "lj"), ("npt", "mixture")))
        case |= {"ensemble": ensemble, "potential": kind,
                 "atoms": _log_int(rng, 320 if ensemble == "nvt" else 1_500,
                                   100_000 if small else 500_000),
                 "skin": rng.choice((0.1, 0.2)), "steps": 50, **box}
    elif path == "md_batch":
        case |= {"systems": rng.randint(3, 12), "low": 320, "high": _log_int(rng, 5_000, 100_000),
                 "skin": rng.choice((0.1, 0.2)), "steps": 50}
    elif path == "evaluate":
        case |= {"atoms": _log_int(rng, 300, 500_000), "order": order,
                 "potential": rng.choice(("lj", "table", "mixture", "sum")), **box}
    elif path == "follow":
        case |= {"atoms": _log_int(rng, 300, 300_000), "order": order,
                 "potential": rng.choice(("lj", "table", "mixture", "sum")),
                 "skin": rng.choice((0.05, 0.1, 0.2)), "frames": rng.randint(3, 6), **box}
    elif path == "differentiate":
        case |= {"atoms": _log_int(rng, 300, 100_000), "order": order,
                 "potential": rng.choice(("lj", "table", "mixture")), **box}
    elif path == "batch":
        case |= {"systems": rng.randint(5, 200), "low": 64, "high": _log_int(rng, 2_000, 30_000)}
    else:
        frames = rng.randint(5, 48)
        case |= {"frames": frames, "atoms": _log_int(rng, 400, 3_000),
                 "batch": rng.choice((frames, max(1, frames // 4))), "updates": rng.randint(10, 60),
                 "potential": rng.choice(("table", "mixture"))}
    return case


# ---- inputs: frames, potentials, velocities --------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _box(atoms, ry, rz, cutoff, density=workloads.DENSITY):
    """The cell's edges at the density, all above twice the cutoff: a small box is nearer to a
    cube, the smallest ones are stretched."""
    for share in (1.0, 0.75, 0.5, 0.25, 0.0):
        ratios = 1.0 + share * np.array([0.0, ry - 1.0, rz - 1.0])
        lengths = ratios * (atoms / density / ratios.prod()) ** (1 / 3)
        if lengths.min() >= 2 * cutoff + 0.05:
            return lengths
    return lengths * (2 * cutoff + 0.05) / lengths.min()


def _positions(atoms, lengths, seed, dtype, jitter=0.02, order="lattice"):
    """A jittered lattice of `atoms` sites spread evenly over one that fills the box."""
    per = np.maximum(1, np.round(lengths / (lengths.prod() / atoms) ** (1 / 3))).astype(int)
    while per.prod() < atoms:
        per[np.argmin(per / lengths)] += 1
    g = _generator(seed)
    site = (torch.arange(atoms, device="cuda") * int(per.prod())) // atoms
    if order == "shuffled":
        site = site[torch.randperm(atoms, generator=g, device="cuda")]
    k = torch.stack((site % int(per[0]), site // int(per[0]) % int(per[1]),
                     site // int(per[0] * per[1])), dim=1).double()
    a = torch.tensor(lengths / per, device="cuda")
    shift = torch.rand((atoms, 3), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    return ((k + 0.5) * a + jitter * shift).to(dtype)


def _cutoff(kind):
    return 1.0 if kind in ("lj", "mixture") else 1.2


def _types(kind, atoms):
    """Atom types [N]: two types, every third atom the second, for a mixture; else all 0."""
    index = torch.arange(atoms, device="cuda")
    return (index % 3 == 2).long() if kind == "mixture" else torch.zeros_like(index)


def _parts(kind, dtype):
    """The parameters of a potential: argon LJ, a 200-knot table, a two-type LJ mixture, or the
    sum of an LJ and a table of half the depth each."""
    def column(values):
        return torch.tensor(values, dtype=dtype, device="cuda")

    sigma, epsilon = workloads.ARGON_SIGMA, workloads.ARGON_EPSILON
    lj = {"sigma": column([sigma]), "epsilon": column([epsilon]), "cutoff": 1.0}
    table = {"table": column(workloads.lj_table(noise=0.0)[None]), "start": column([0.3]), "cutoff": 1.2}
    mixture = {"sigma": column([sigma, 0.35, 0.36]), "epsilon": column([epsilon, 1.15, 1.33]),
               "cutoff": 1.0}
    half = column(workloads.lj_table(noise=0.0, epsilon=epsilon / 2)[None])
    return {"lj": [lj], "table": [table], "mixture": [mixture],
            "sum": [dict(lj, epsilon=column([epsilon / 2]), cutoff=0.9),
                    dict(table, table=half)]}[kind]


def _model(parts, types, trainable=False):
    models = []
    for part in parts:
        if "table" in part:
            models.append(potential.tabulated(atom_types=types, **part,
                                              trainable=("table",) if trainable else ()))
        else:
            names = ("sigma", "epsilon") if trainable else ()
            models.append(potential.lennard_jones(atom_types=types, **part, trainable=names))
    return models[0] if len(models) == 1 else potential.sum(*models)


def _dtype(case):
    return getattr(torch, case["dtype"])


def _system(case, seed):
    """Positions, cell, parameters and types of a one-system case."""
    n, dtype = case["atoms"], _dtype(case)
    lengths = _box(n, case["ry"], case["rz"], _cutoff(case["potential"]))
    x = _positions(n, lengths, seed, dtype, order=case.get("order", "lattice"))
    return (x, torch.tensor(lengths, dtype=dtype, device="cuda"),
            _parts(case["potential"], dtype), _types(case["potential"], n))


def _motion(types, seed, dtype):
    masses = torch.full(types.shape, workloads.ARGON_MASS, dtype=dtype, device="cuda")
    masses[types == 1] = 83.798
    return masses, md.maxwell_boltzmann(masses, 120.0, int(seed))


def _sizes(case):
    """The systems' sizes: the range's logarithm cut evenly, in a fixed mixed order."""
    count, low, high = case["systems"], case["low"], case["high"]
    sizes = [int(low * (high / low) ** ((k + 0.5) / count)) + k % 2 for k in range(count)]
    random.Random(count).shuffle(sizes)
    return sizes


def _many(case, seed):
    """(positions, cell, parts, types) of each system, LJ and tables in turn."""
    out = []
    for k, n in enumerate(_sizes(case)):
        shape = random.Random(1000 * case["systems"] + k)
        kind = ("lj", "table")[k % 2]
        out.append(_system({"atoms": n, "potential": kind, "dtype": case["dtype"],
                            "ry": shape.uniform(1, 2), "rz": shape.uniform(1, 2)},
                           int(seed) * 1000 + k))
    return out


def _follow_frames(case, seed):
    """Consecutive frames 16 fs apart, the atoms flying at 120 K."""
    x, cell, parts, types = _system(case, seed)
    _, v = _motion(types, seed, x.dtype)
    return [x + (_SPACING * k) * v for k in range(case["frames"])], cell, parts, types


def _restraint(x, anchors):
    return 50.0 * (x - anchors).square().sum()


def _fit_data(case, seed):
    """Frames [F, N, 3], cells [F, 3], types, the labels of a hidden LJ model (the forces with
    noise) and the parameters that the fit starts from."""
    frames, n, dtype = case["frames"], case["atoms"], _dtype(case)
    lengths = _box(n, 1.0, 1.0, 1.2, density=8.0)
    x = torch.stack([_positions(n, lengths, int(seed) * 1000 + f, dtype, jitter=0.05)
                     for f in range(frames)])
    cell = torch.tensor(lengths, dtype=dtype, device="cuda")
    types = _types(case["potential"], n)
    two = case["potential"] == "mixture"
    truth = {"sigma": torch.tensor([0.47, 0.46, 0.45][:3 if two else 1], device="cuda").double(),
             "epsilon": torch.tensor([3.5, 3.2, 3.0][:3 if two else 1], device="cuda").double(),
             "cutoff": 1.2}
    wide, box = x.double(), cell.double()
    e, f, w = _frames_efw(_frames_geometry(_frame_pairs(wide, box, 1.2), wide, box, types,
                                           range(frames)), truth)
    noise = torch.randn(f.shape, generator=_generator(seed), device="cuda", dtype=torch.float64)
    labels = {"energy": e.to(dtype), "forces": (f + 5.0 * noise).to(dtype), "virial": w.to(dtype)}
    if two:
        start = {"sigma": truth["sigma"].to(dtype) * 0.97, "epsilon": truth["epsilon"].to(dtype) * 0.9,
                 "cutoff": 1.2}
    else:
        r = np.linspace(0.3, 1.2, 200)
        s6 = (0.45 / r) ** 6
        knots = np.clip(4 * 3.0 * (s6 * s6 - s6), -50, 50)
        knots[-1] = 0.0
        start = {"table": torch.tensor(knots[None], dtype=dtype, device="cuda"),
                 "start": torch.tensor([0.3], dtype=dtype, device="cuda"), "cutoff": 1.2}
    return x, cell.expand(frames, 3).contiguous(), types, labels, start


def _rate(case):
    return 1e-2 if case["potential"] == "table" else 1e-3


# ---- prepare and run -------------------------------------------------------------------------


def prepare(case, seed):
    return {"md": _prepare_md, "md_batch": _prepare_md_batch, "evaluate": _prepare_evaluate,
            "follow": _prepare_follow, "differentiate": _prepare_differentiate,
            "batch": _prepare_batch, "fit": _prepare_fit}[case["path"]](case, seed)


def run(state):
    return state["pass"](state)


def _prepare_md(case, seed):
    x, cell, parts, types = _system(case, seed)
    masses, v = _motion(types, seed, x.dtype)
    settings = {"timestep": _TIMESTEP, "temperature": 120.0, "thermostat_timescale": _TAU,
                "skin": case["skin"]}
    if case["ensemble"] == "npt":
        sim = md.npt(_model(parts, types), x, v, masses, cell, pressure=750 * units.BAR,
                     barostat_timescale=1.0, **settings)
    else:
        sim = md.nvt(_model(parts, types), x, v, masses, cell, **settings)
    return {"pass": _run_md, "simulation": sim, "steps": case["steps"]}


def _frame(sim):
    s = sim.state()
    return {"positions": s.positions, "velocities": s.velocities, "forces": s.forces,
            "images": s.images, "cell": s.cell}


def _run_md(state):
    state["simulation"].run(state["steps"])
    return _frame(state["simulation"])


def _prepare_md_batch(case, seed):
    sims, kinds = [], {}
    for k, (x, cell, parts, types) in enumerate(_many(case, seed)):
        masses, v = _motion(types, int(seed) * 1000 + k, x.dtype)
        sims.append(md.Simulation(
            _model(parts, types), x, v, masses, cell, timestep=_TIMESTEP, skin=case["skin"],
            capacity_multiplier=1.25, images=None, step=0, temperature=120.0,
            thermostat_timescale=_TAU, force_group=4, graphs=False))
        kinds.setdefault("table" in parts[0], []).append(sims[-1])
    batches = [md.SimulationBatch(group) for group in kinds.values()]
    return {"pass": _run_md_batch, "simulations": sims, "batches": batches,
            "streams": [torch.cuda.Stream() for _ in batches], "steps": case["steps"]}


def _run_md_batch(state):
    here = torch.cuda.current_stream()
    for batch, stream in zip(state["batches"], state["streams"]):
        stream.wait_stream(here)
        with torch.cuda.stream(stream):
            batch.advance(state["steps"])
    for stream in state["streams"]:
        here.wait_stream(stream)
    for sim in state["simulations"]:
        sim.check()
    return [{k: v for k, v in _frame(sim).items() if k != "cell"} for sim in state["simulations"]]


def _prepare_evaluate(case, seed):
    x, cell, parts, types = _system(case, seed)
    model = _model(parts, types)
    inner = tuple(p["cutoff"] for p in parts[:-1])
    return {"pass": _run_evaluate, "positions": x, "cell": cell, "model": model,
            "inner": inner, "efw": quantity.energy_force_virial(model)}


def _run_evaluate(state):
    x, cell = state["positions"], state["cell"]
    pairs = NeighborList(state["model"].cutoff, inner_cutoffs=state["inner"])
    pairs.allocate(x, cell)
    e, f, w = state["efw"](x, cell, pairs.tensors())
    return {"energy": e, "forces": f, "virial": w}


def _prepare_follow(case, seed):
    frames, cell, parts, types = _follow_frames(case, seed)
    model = _model(parts, types)
    pairs = NeighborList(model.cutoff, skin=case["skin"],
                         inner_cutoffs=tuple(p["cutoff"] for p in parts[:-1]))
    pairs.allocate(frames[0], cell)
    return {"pass": _run_follow, "frames": frames, "cell": cell, "list": pairs,
            "efw": quantity.energy_force_virial(model)}


def _run_follow(state):
    out = []
    for x in state["frames"][1:] + state["frames"][:1]:
        state["list"].update(x, state["cell"])
        out.append(state["efw"](x, state["cell"], state["list"].tensors()))
    return out


def _prepare_differentiate(case, seed):
    x, cell, parts, types = _system(case, seed)
    model = _model(parts, types, trainable=True)
    anchors = _positions(x.shape[0], cell.double().cpu().numpy(), int(seed) + 1, x.dtype,
                         order="lattice")
    pairs = NeighborList(model.cutoff)
    pairs.allocate(x, cell)

    def energy(positions, box, listed_pairs, strain=None):
        return model(positions, box, listed_pairs, strain) + _restraint(positions, anchors)

    return {"pass": _run_differentiate, "positions": x, "cell": cell, "model": model,
            "pairs": pairs.tensors(), "efw": quantity.energy_force_virial(energy)}


def _run_differentiate(state):
    x, cell, pairs = state["positions"], state["cell"], state["pairs"]
    e, f, w = state["efw"](x, cell, pairs)
    slopes = torch.autograd.grad(state["model"](x, cell, pairs), tuple(state["model"].parameters()))
    return {"energy": e, "forces": f, "virial": w, "parameters": slopes}


def _prepare_batch(case, seed):
    systems = _many(case, seed)
    batch = Batch([(x, cell, _model(parts, types)) for x, cell, parts, types in systems])
    batch.evaluate()
    moved = [s[0] for s in _many(case, int(seed) + 500_000)]
    return {"pass": _run_batch, "batch": batch, "frames": moved}


def _run_batch(state):
    state["batch"].set_positions(state["frames"])
    e, f, w = state["batch"].evaluate()
    return {"energy": e, "forces": f, "virial": w}


def _prepare_fit(case, seed):
    x, cells, types, labels, start = _fit_data(case, seed)
    data = training.Dataset(x, cells, **labels)
    return {"pass": _run_fit, "data": data, "start": start, "types": types,
            "updates": case["updates"], "batch": case["batch"], "rate": _rate(case)}


def _run_fit(state):
    model = _model([state["start"]], state["types"], trainable=True)
    optimizer = torch.optim.Adam(model.parameters(), lr=state["rate"])
    training.fit(model, state["data"], optimizer, updates=state["updates"],
                 batch_size=state["batch"], energy=1.0, forces=1.0, virial=1.0)
    return [p.detach() for p in model.parameters()]


# ---- what a pass cannot do without -----------------------------------------------------------


def _pair_count(atoms, cutoff, density=workloads.DENSITY):
    return atoms * density * 4 / 3 * math.pi * cutoff**3 / 2


def _pair_flops(kind):
    """Distance with its periodic image, the terms, and both atoms' force and virial sums."""
    return {"lj": 45, "mixture": 47, "table": 60, "sum": 90}[kind]


def work(case):
    s = 8 if case["dtype"] == "float64" else 4
    path = case["path"]
    if path in ("md", "md_batch"):
        # each step: positions and velocities read and written, forces read and written, masses
        one = [(case["atoms"], case["potential"])] if path == "md" else list(
            zip(_sizes(case), ("lj", "table") * case["systems"]))
        atoms = sum(n for n, _ in one)
        flops = sum(_pair_count(n, _cutoff(k)) * _pair_flops(k) + 40 * n for n, k in one)
        return {"bytes": case["steps"] * atoms * 19 * s, "flops": case["steps"] * flops}
    if path == "batch":
        one = list(zip(_sizes(case), ("lj", "table") * case["systems"]))
        return {"bytes": sum(n for n, _ in one) * 6 * s,
                "flops": sum(_pair_count(n, _cutoff(k)) * _pair_flops(k) for n, k in one)}
    if path == "fit":
        pairs = case["frames"] * _pair_count(case["atoms"], 1.2, 8.0)
        atoms = case["frames"] * case["atoms"]
        share = case["batch"] / case["frames"] * case["updates"]
        # per update: positions and force labels read, the pairs met twice (values, gradients)
        return {"bytes": share * atoms * 6 * s + 8 * pairs, "flops": share * pairs * 120}
    cutoff, atoms = _cutoff(case["potential"]), case["atoms"]
    pairs, each = _pair_count(atoms, cutoff), _pair_flops(case["potential"])
    if path in ("evaluate", "follow"):  # positions in, forces out
        frames = case.get("frames", 1)
        return {"bytes": frames * atoms * 6 * s, "flops": frames * pairs * each}
    return {"bytes": atoms * 9 * s + 8 * pairs, "flops": 2 * pairs * each}


# ---- the same in 64 bits, by plain torch -----------------------------------------------------


def _separation(x, i, j, cell):
    d = x[i] - x[j]
    return d - cell * torch.round(d / cell)


def _pairs(x, cell, radius):
    """Pairs (i, j) [2, P] closer than the radius, each once: every pair in a small or narrow
    system, else cells of the radius against half of their neighbors."""
    n = x.shape[0]
    dims = [int(L // radius) for L in cell.tolist()]
    found = []
    if n <= 4096 or min(dims) < 3:
        index = torch.arange(n, device=x.device)
        for rows in index.split(max(1, 40_000_000 // n)):
            d = x[rows, None, :] - x[None, :, :]
            d -= cell * torch.round(d / cell)
            hit = (d.square().sum(-1) < radius**2) & (index[None, :] > rows[:, None])
            a, b = hit.nonzero(as_tuple=True)
            found.append(torch.stack((rows[a], b)))
        return torch.cat(found, dim=1)
    nx, ny, nz = dims
    count = torch.tensor(dims, device=x.device)
    home = (torch.remainder(x, cell) / cell * count).long().clamp(min=0)
    home = torch.minimum(home, count - 1)
    cell_of = home[:, 0] + nx * (home[:, 1] + ny * home[:, 2])
    order = torch.argsort(cell_of)
    held = torch.bincount(cell_of, minlength=nx * ny * nz)
    first = held.cumsum(0) - held
    rank = torch.arange(n, device=x.device) - first[cell_of[order]]
    members = torch.full((nx * ny * nz, int(held.max())), -1, dtype=torch.long, device=x.device)
    members[cell_of[order], rank] = order
    steps = [(sx, sy, sz) for sz in (-1, 0, 1) for sy in (-1, 0, 1) for sx in (-1, 0, 1)]
    room = members.shape[1] ** 2
    for cells in torch.arange(nx * ny * nz, device=x.device).split(max(1, 40_000_000 // room)):
        cx, cy, cz = cells % nx, cells // nx % ny, cells // (nx * ny)
        for sx, sy, sz in steps[13:]:
            other = (cx + sx) % nx + nx * ((cy + sy) % ny + ny * ((cz + sz) % nz))
            a, b = members[cells][:, :, None], members[other][:, None, :]
            d = x[a] - x[b]
            d -= cell * torch.round(d / cell)
            hit = (d.square().sum(-1) < radius**2) & (a >= 0) & (b >= 0)
            if (sx, sy, sz) == (0, 0, 0):
                hit &= b > a
            k, p, q = hit.nonzero(as_tuple=True)
            found.append(torch.stack((members[cells[k], p], members[other[k], q])))
    return torch.cat(found, dim=1)


def _pair_terms(part, row, r2):
    """A pair's energy and -(du/dr)/r within the part's cutoff, 0 beyond it."""
    inside = r2 < part["cutoff"] ** 2
    if "table" in part:
        knots = part["table"].double()
        start = part["start"].double()[row]
        count = knots.shape[1]
        spacing = (part["cutoff"] - part["start"].double()) / (count - 1)
        h = spacing[row]
        v = torch.cat((knots[:, :-1], torch.zeros_like(knots[:, :1])), dim=1)
        v = torch.cat((3 * v[:, :1] - 3 * v[:, 1:2] + v[:, 2:3], v,
                       3 * v[:, -1:] - 3 * v[:, -2:-1] + v[:, -3:-2]), dim=1).reshape(-1)
        r = r2.sqrt()
        at = (r - start) / h
        segment = at.floor().clamp(0, count - 2)
        t = at - segment
        base = row * (count + 2) + segment.long()
        u0, u1, u2, u3 = (v[base + k] for k in range(4))
        a, b, c = u2 - u0, 2 * u0 - 5 * u1 + 4 * u2 - u3, 3 * (u1 - u2) + u3 - u0
        s, below = t.clamp(min=0), t.clamp(max=0)
        u = u1 + 0.5 * s * (a + s * (b + s * c)) + 0.5 * a * below
        slope = 0.5 * (a + s * (2 * b + 3 * s * c))
        fs = -slope / h / r
    else:
        s2, eps = part["sigma"].double()[row].square(), part["epsilon"].double()[row]
        p, q = (s2 / r2) ** 3, (s2 / part["cutoff"] ** 2) ** 3
        u = 4 * eps * (p * p - p - (q * q - q))
        fs = 24 * eps * (2 * p * p - p) / r2
    return torch.where(inside, u, 0.0), torch.where(inside, fs, 0.0)


def _rows(types, i, j):
    return types[i] + types[j]  # two types at most: rows (0, 0), (0, 1), (1, 1)


def _gather_sums(pairs, atoms):
    """What ``_atom_sums`` needs to add a pair's vector to its first atom and take it from its
    second: both orientations sorted by atom, and where each atom's run ends."""
    order = torch.argsort(torch.cat((pairs[0], pairs[1])))
    ends = torch.bincount(pairs.reshape(-1), minlength=atoms).cumsum(0)
    return order, ends


def _atom_sums(g, order, ends):
    """[N, 3] sums of the pairs' vectors g [P, 3] per atom, by differences of running sums."""
    running = torch.cat((g.t(), -g.t()), dim=1)[:, order].cumsum(dim=1)
    running = torch.cat((torch.zeros_like(running[:, :1]), running), dim=1)
    starts = torch.cat((torch.zeros_like(ends[:1]), ends[:-1]))
    return (running[:, ends] - running[:, starts]).t().contiguous()


def _efw(pairs, x, cell, parts, types, sums=None):
    i, j = pairs
    d = _separation(x, i, j, cell)
    r2, row = d.square().sum(-1), _rows(types, i, j)
    terms = [_pair_terms(part, row, r2) for part in parts]
    fs = sum(t[1] for t in terms)
    g = fs[:, None] * d
    forces = _atom_sums(g, *(_gather_sums(pairs, x.shape[0]) if sums is None else sums))
    virial = torch.stack([(d[:, a] * g[:, b]).sum() for a in range(3) for b in range(3)])
    return sum(t[0].sum() for t in terms), forces, virial.view(3, 3)


def _frame_pairs(x, cell, radius):
    """Each frame's pairs, the atoms of frame f numbered from f N."""
    n = x.shape[1]
    return [_pairs(x[f], cell, radius) + f * n for f in range(x.shape[0])]


def _frames_geometry(pairs, x, cell, types, chosen):
    """The chosen frames' pair vectors, parameter rows, counts and sums per atom."""
    n = x.shape[1]
    index = torch.cat([pairs[f] - (f - k) * n for k, f in enumerate(chosen)], dim=1)
    i, j = index
    d = _separation(x[list(chosen)].reshape(-1, 3), i, j, cell)
    return {"d": d, "r2": d.square().sum(-1), "row": _rows(types, i % n, j % n),
            "counts": [pairs[f].shape[1] for f in chosen],
            "sums": _gather_sums(index, len(chosen) * n)}


def _frames_efw(geometry, part):
    """E [B], F [B, N, 3] and W [B, 3, 3] of frames, differentiable in the part's parameters."""
    d, counts = geometry["d"], geometry["counts"]
    u, fs = _pair_terms(part, geometry["row"], geometry["r2"])
    g = fs[:, None] * d
    forces = _atom_sums(g, *geometry["sums"]).view(len(counts), -1, 3)
    energy = torch.stack([v.sum() for v in u.split(counts)])
    virial = torch.stack([a.t() @ b for a, b in zip(d.split(counts), g.split(counts))])
    return energy, forces, virial


def _chain_half(kinetic, q, p, masses, g):
    """Half a step of a Nose-Hoover chain of 3: the velocities' factor and the moved chain."""
    quarter, eighth = 0.25 * _TIMESTEP, 0.125 * _TIMESTEP

    def drive(k):
        return 2 * kinetic - g * _KT if k == 0 else p[k - 1] ** 2 / masses[k - 1] - _KT

    damp = [None, None]
    p = list(p)
    for k in (2, 1, 0):
        p[k] = (p[k] + quarter * drive(k) if k == 2
                else damp[k] * (damp[k] * p[k] + quarter * drive(k)))
        if k > 0:
            damp[k - 1] = torch.exp(-eighth * p[k] / masses[k])
    factor = torch.exp(-0.5 * _TIMESTEP * p[0] / masses[0])
    kinetic = kinetic * factor**2
    q = [q[k] + 0.5 * _TIMESTEP * p[k] / masses[k] for k in range(3)]
    for k in (0, 1, 2):
        p[k] = (p[k] + quarter * drive(k) if k == 2
                else damp[k] * (damp[k] * p[k] + quarter * drive(k)))
    return factor, q, p


def _nvt(x, cell, parts, types, masses, v, steps):
    """Velocities and forces after `steps` of velocity Verlet with a Nose-Hoover chain of 3."""
    x, cell, masses, v = x.double(), cell.double(), masses.double(), v.double()
    reach = max(p["cutoff"] for p in parts) + 0.15
    column = masses[:, None]
    v = v - (column * v).sum(0) / masses.sum()
    g = 3 * x.shape[0] - 3
    chain = [g * _KT * _TAU**2, _KT * _TAU**2, _KT * _TAU**2]
    zero = torch.zeros((), dtype=torch.float64, device=x.device)
    q, p = [zero] * 3, [zero] * 3
    pairs = _pairs(x, cell, reach)
    sums = _gather_sums(pairs, x.shape[0])
    forces = _efw(pairs, x, cell, parts, types, sums)[1]
    for step in range(1, steps + 1):
        kinetic = 0.5 * (column * v.square()).sum()
        factor, q, p = _chain_half(kinetic, q, p, chain, g)
        v = v * factor + 0.5 * _TIMESTEP * forces / column
        x = x + _TIMESTEP * v
        if step % 10 == 0:
            pairs = _pairs(x, cell, reach)
            sums = _gather_sums(pairs, x.shape[0])
        forces = _efw(pairs, x, cell, parts, types, sums)[1]
        v = v + 0.5 * _TIMESTEP * forces / column
        factor, q, p = _chain_half(0.5 * (column * v.square()).sum(), q, p, chain, g)
        v = v * factor
    return v, forces


def _exact_frame(system, seed, steps):
    # positions and images change by a whole edge where an atom lies on a face: no exact value
    x, cell, parts, types = system
    masses, v = _motion(types, seed, x.dtype)
    v, forces = _nvt(x, cell, parts, types, masses, v, steps)
    return {"positions": None, "velocities": v, "forces": forces, "images": None}


def exact(case, seed):
    path = case["path"]
    if path == "md":
        if case["ensemble"] == "npt" or case["atoms"] * case["steps"] > 4_000_000:
            return None
        system = _system(case, seed)
        return _exact_frame(system, seed, case["steps"]) | {"cell": system[1].double()}
    if path == "md_batch":
        return [_exact_frame(system, int(seed) * 1000 + k, case["steps"])
                for k, system in enumerate(_many(case, seed))]
    if path == "fit":
        return _exact_fit(case, seed)
    if path == "batch":
        found = []
        for (_, cell, parts, types), moved in zip(_many(case, seed),
                                                  _many(case, int(seed) + 500_000)):
            x, box = moved[0].double(), cell.double()
            found.append(_efw(_pairs(x, box, parts[0]["cutoff"]), x, box, parts, types))
        e, f, w = zip(*found)
        return {"energy": torch.stack(e), "forces": torch.cat(f), "virial": torch.stack(w)}
    if path == "follow":
        frames, cell, parts, types = _follow_frames(case, seed)
    else:
        x, cell, parts, types = _system(case, seed)
        frames = [x]
    box, reach = cell.double(), max(p["cutoff"] for p in parts)
    if path == "differentiate":
        return _exact_differentiate(frames[0], box, parts, types, seed)
    found = []
    for x in frames[1:] + frames[:1]:
        x = x.double()
        found.append(_efw(_pairs(x, box, reach), x, box, parts, types))
    if path == "follow":
        return found
    e, f, w = found[0]
    return {"energy": e, "forces": f, "virial": w}


def _exact_differentiate(x, box, parts, types, seed):
    anchors = _positions(x.shape[0], box.cpu().numpy(), int(seed) + 1, x.dtype).double()
    names = ["table"] if "table" in parts[0] else ["sigma", "epsilon"]
    part = dict(parts[0])
    for name in names:
        part[name] = part[name].double().requires_grad_(True)
    x = x.double()
    e, f, w = _efw(_pairs(x, box, part["cutoff"]), x, box, [part], types)
    slopes = torch.autograd.grad(e, [part[name] for name in names])
    e, f, w = e.detach(), f.detach(), w.detach()
    return {"energy": e + _restraint(x, anchors), "forces": f - 100.0 * (x - anchors),
            "virial": w, "parameters": list(slopes)}


def _exact_fit(case, seed):
    x, cells, types, labels, start = _fit_data(case, seed)
    x, box = x.double(), cells[0].double()
    labels = {k: v.double() for k, v in labels.items()}
    pairs = _frame_pairs(x, box, 1.2)
    scale = {k: (v - v.mean(0) if k != "forces" else v).square().mean().sqrt()
             for k, v in labels.items()}
    part = {k: v.double() if torch.is_tensor(v) else v for k, v in start.items()}
    names = ["table"] if "table" in part else ["sigma", "epsilon"]
    for name in names:
        part[name] = part[name].clone().requires_grad_(True)
    optimizer = torch.optim.Adam([part[name] for name in names], lr=_rate(case))
    generator, order = torch.Generator().manual_seed(0), []
    while len(order) < case["updates"]:
        order.extend(torch.randperm(case["frames"], generator=generator).split(case["batch"]))
    geometry, held = None, None
    for chosen in order[:case["updates"]]:
        chosen = sorted(chosen.tolist())
        if chosen != held:
            geometry, held = _frames_geometry(pairs, x, box, types, chosen), chosen
        found = dict(zip(("energy", "forces", "virial"), _frames_efw(geometry, part)))
        loss = sum(((found[k] - labels[k][chosen]) / scale[k]).square().mean() for k in found)
        optimizer.zero_grad()
        loss.backward()
        optimizer.step()
    return [part[name].detach() for name in names]
