"""The work that users of this library have it do, as cases that can be timed and compared: neighbor lists of single
systems from a few hundred atoms to a million, lists on host arrays, batches of small systems, the steps of a
trajectory with a skin, and neighbor lists with the gradient that turns them into forces.

Rows of a list with ``sorted=True`` come in the same order on every run and are returned as they are. Rows of an
unsorted single system come in order of arrival, so what is returned of those calls is what their user computes from
them: energy, forces and virial, which do not depend on that order. (Batches of free molecules have an order of their
own also when they are not sorted.)
"""

import math

import numpy as np
import torch

from vesin_amd import NeighborList

DIAMOND_A = 3.567  # edge of the 8-atom cell of carbon, in Angstrom
DIAMOND_BASIS = [
    [0.0, 0.0, 0.0], [0.0, 0.5, 0.5], [0.5, 0.0, 0.5], [0.5, 0.5, 0.0],
    [0.25, 0.25, 0.25], [0.25, 0.75, 0.75], [0.75, 0.25, 0.75], [0.75, 0.75, 0.25],
]
BYTES_OF = {"P": 16, "S": 12, "d": 8, "D": 24}
ROWS_AT_MOST = 60_000_000  # of a drawn case; the largest listed ones have 89 and 190 million

# ---- the cases

# kind "list": one call of NeighborList.compute; "host": the same on numpy arrays; "batch": compute_batch on the
# batches of a loader, one after the other; "trajectory": one call per frame with a skin; "forces": the TorchScript
# class with the gradient of the distances (and vectors) with respect to points (and box).


def listed():
    return [
        # latency: a small supercell that is searched again and again (relaxations, Monte Carlo moves, small MD)
        dict(name="supercell-216", kind="list", system="diamond", replicas=3, shuffled=False, cutoff=5.0, full=True, sorted=True,
             quantities="PSd", dtype="float64"),
        # the numpy caller: scripts around ASE and descriptors of single structures
        dict(name="host-1728", kind="host", system="diamond", replicas=6, shuffled=False, cutoff=5.0, full=True, sorted=True,
             quantities="ijSd", dtype="float64"),
        # an everyday MD box, single precision as ML potentials use it, half list with vectors
        dict(name="liquid-10k", kind="list", system="liquid", points=10_007, density=0.1, skew=0.0, periodic=7, cutoff=6.0,
             full=False, sorted=True, quantities="PSdD", dtype="float32"),
        # a large triclinic box at liquid density
        dict(name="triclinic-100k", kind="list", system="liquid", points=100_000, density=0.1, skew=0.3, periodic=7, cutoff=6.0,
             full=False, sorted=True, quantities="PSdD", dtype="float64"),
        # the headline system, sorted for reproducible training and for CSR graphs
        dict(name="diamond-1M", kind="list", system="diamond", replicas=50, shuffled=False, cutoff=5.0, full=True, sorted=True,
             quantities="PSd", dtype="float64"),
        # uneven density: clusters without periodic directions (aerosols, aggregates, point clouds)
        dict(name="clusters-500k", kind="list", system="clusters", points=500_000, blobs=50, periodic=0, cutoff=4.5, full=True,
             sorted=True, quantities="Pd", dtype="float64"),
        # one step of a pair potential: neighbor list of the headline system and its forces
        dict(name="forces-1M", kind="forces", system="diamond", replicas=50, shuffled=False, cutoff=5.0, full=True, sorted=False,
             quantities="d", box_gradient=False, dtype="float64"),
        # one training step on a mid-size box: distances and vectors in single precision, forces and virial
        dict(name="virial-50k", kind="forces", system="liquid", points=50_021, density=0.08, skew=0.2, periodic=7, cutoff=5.0,
             full=True, sorted=False, quantities="dD", box_gradient=True, dtype="float32"),
        # thousands of replicas of a cell smaller than the cutoff (sampling, phonons)
        dict(name="replicas-4096", kind="batch", system="replicas", systems=4096, replicas=2, batches=1, cutoff=10.0, full=True,
             sorted=True, quantities="PSd"),
        # a loader of molecules: other ones in every batch
        dict(name="molecules-20k", kind="batch", system="molecules", systems=20_000, smallest=3, largest=40, batches=2, cutoff=5.0,
             full=True, sorted=False, quantities="PdD"),
        # a loader of crystals: other ones in every batch
        dict(name="crystals-2k", kind="batch", system="crystals", systems=2_000, smallest=8, largest=64, batches=2, cutoff=5.0,
             full=True, sorted=True, quantities="PSD"),
        # molecular dynamics with a skin: most steps filter what is kept
        dict(name="trajectory-13824", kind="trajectory", system="diamond", replicas=12, shuffled=False, frames=12, speed=0.006,
             cutoff=5.0, skin=0.5, full=True, sorted=True, quantities="PSd", dtype="float64"),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _draw(rng):
    kind = rng.choice(["list", "list", "list", "host", "forces", "forces", "batch", "batch", "trajectory"])
    case = dict(kind=kind)
    if kind == "batch":
        system = rng.choice(["replicas", "molecules", "crystals"])
        case.update(system=system, batches=1 if system == "replicas" else 2, cutoff=round(rng.uniform(3.5, 6.5), 3),
                    full=rng.random() < 0.7, sorted=system != "molecules" or rng.random() < 0.5,
                    quantities=rng.choice(["PS", "PSd", "PSD", "PSdD"]))
        if system == "replicas":
            case.update(systems=int(_log_uniform(rng, 16, 4096)), replicas=rng.randint(1, 3), cutoff=round(rng.uniform(4.0, 10.0), 3))
        elif system == "molecules":
            case.update(systems=int(_log_uniform(rng, 64, 50_000)), smallest=rng.randint(2, 9), largest=rng.randint(10, 64))
        else:
            case.update(systems=int(_log_uniform(rng, 16, 8_000)), smallest=rng.randint(1, 12), largest=rng.randint(16, 200))
        return case
    case.update(
        cutoff=round(rng.uniform(3.5, 7.0), 3), full=rng.random() < 0.6, sorted=kind != "forces" or rng.random() < 0.3,
        quantities=rng.choice(["P", "PS", "PSd", "PSD", "PSdD"]), dtype="float64" if rng.random() < 0.7 else "float32",
    )
    if kind == "trajectory":
        case.update(system="diamond", replicas=rng.randint(3, 14), shuffled=rng.random() < 0.5, frames=12,
                    speed=round(rng.uniform(0.003, 0.007), 4), skin=0.5)
        return case
    largest = {"list": 1_000_000, "host": 20_000, "forces": 1_000_000}[kind]
    smallest = {"list": 30, "host": 30, "forces": 200}[kind]
    if kind == "forces":
        case.update(quantities=rng.choice(["d", "D", "dD"]), box_gradient=rng.random() < 0.5)
    points = int(_log_uniform(rng, smallest, largest))
    system = rng.choice(["liquid", "liquid", "diamond", "clusters"])
    if system == "clusters" and points >= 2_000:
        case.update(system=system, points=points, blobs=max(1, points // 10_000), periodic=rng.choice([0, 3]), box_gradient=False)
        if kind != "forces":
            del case["box_gradient"]
    elif system == "diamond":
        case.update(system=system, replicas=max(2, round((points / 8) ** (1 / 3))), shuffled=rng.random() < 0.5)
    else:
        case.update(system="liquid", points=points, density=round(_log_uniform(rng, 0.02, 0.15), 4),
                    skew=round(rng.uniform(0.0, 0.4), 3), periodic=rng.choice([7, 7, 7, 3, 0]))
        if case["periodic"] == 0 and kind == "forces":
            case["box_gradient"] = False
    return case


def draw(rng):
    while True:
        case = _draw(rng)
        if _rows(case) * case.get("batches", 1) * case.get("frames", 1) <= ROWS_AT_MOST:
            return case


# ---- inputs

# A case has one structure (one data set, for the batches), whose list has a number of rows of its own. Another seed is
# another frame of it, with other coordinates and other labels and as many rows: the points are moved, turned around,
# and numbered in another order, the systems of a batch are shuffled. Points in single precision are multiples of
# 2^-12, like the decimals of a file, so that moving them keeps every distance.

GRID = 4096.0


def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    return generator


def _random(generator, *shape):
    return torch.rand(shape, device="cuda", dtype=torch.float64, generator=generator)


def _normal(generator, *shape):
    return torch.randn(shape, device="cuda", dtype=torch.float64, generator=generator)


def _lattice(replicas):
    cells = torch.cartesian_prod(*[torch.arange(replicas, device="cuda", dtype=torch.float64)] * 3).reshape(-1, 3)
    basis = torch.tensor(DIAMOND_BASIS, device="cuda", dtype=torch.float64)
    return (cells[:, None, :] + basis[None, :, :]).reshape(-1, 3) * DIAMOND_A


def _box_shape(skew):
    """Edges of 1, 1.05 and 1.1, sheared by ``skew``, scaled to unit volume."""
    box = torch.tensor([[1.0, 0.0, 0.0], [skew * 0.6, 1.05, 0.0], [skew, skew * 0.4, 1.1]], dtype=torch.float64)
    return box / torch.det(box) ** (1.0 / 3.0)


def _structure(case):
    """(points, velocities, box, three flags, points per window that the order of the points is kept outside of)."""
    generator = _generator(7)
    if case["system"] == "diamond":
        points = _lattice(case["replicas"])
        points = points + 0.05 * _normal(generator, *points.shape)
        box = torch.eye(3, dtype=torch.float64, device="cuda") * (case["replicas"] * DIAMOND_A)
        periodic, window = 7, len(points) if case["shuffled"] else 8
    elif case["system"] == "liquid":
        box = (_box_shape(case["skew"]) * (case["points"] / case["density"]) ** (1.0 / 3.0)).cuda()
        points = _random(generator, case["points"], 3) @ box
        periodic, window = case["periodic"], case["points"]
    else:
        edge = 300.0 * (case["blobs"] / 50) ** (1.0 / 3.0)
        centres = _random(generator, case["blobs"], 3) * edge
        which = torch.randint(0, case["blobs"], (case["points"],), device="cuda", generator=generator)
        points = centres[which] + 8.0 * _normal(generator, case["points"], 3)
        box = torch.eye(3, dtype=torch.float64, device="cuda") * edge
        periodic, window = case["periodic"], case["points"]
    velocities = case.get("speed", 0.0) * _normal(generator, *points.shape)
    return points, velocities, box, [bool(periodic >> axis & 1) for axis in range(3)], window


def _single_system(case, seed):
    """The frames of a case (all but trajectories have one), its box and its three flags."""
    points, velocities, box, periodic, window = _structure(case)
    grid = GRID if case["dtype"] == "float32" else None
    if grid is not None:
        box = torch.round(box * grid) / grid
    generator = _generator(seed)
    offset = torch.floor(_random(generator, 3) * GRID) / GRID
    turned = bool(torch.randint(0, 2, (1,), device="cuda", generator=generator).item())
    positions = torch.arange(len(points), device="cuda")
    order = torch.argsort(positions // window + _random(generator, len(points)))
    frames = []
    for step in range(case.get("frames", 1)):
        frame = points + step * velocities
        if grid is not None:
            frame = torch.round(frame * grid) / grid
        frame = (box.sum(dim=0) - frame if turned else frame) + offset
        frames.append(frame[order].to(getattr(torch, case["dtype"])).contiguous())
    return frames, box.to(getattr(torch, case["dtype"])), periodic


def _batch(case, number, seed):
    """One batch of the data set: (points, first_point, boxes, periodic)."""
    n_systems = case["systems"]
    generator = _generator(11 + number)
    if case["system"] == "replicas":
        lattice = _lattice(case["replicas"])
        sizes = np.full(n_systems, len(lattice))
    else:
        sizes = np.random.default_rng(11 + number).integers(case["smallest"], case["largest"] + 1, n_systems)
    n_of = torch.as_tensor(sizes, device="cuda")
    system_of = torch.repeat_interleave(torch.arange(n_systems, device="cuda"), n_of)
    if case["system"] == "replicas":
        boxes = torch.eye(3, dtype=torch.float64, device="cuda").repeat(n_systems, 1, 1) * (case["replicas"] * DIAMOND_A)
        points = lattice.repeat(n_systems, 1) + 0.05 * _normal(generator, len(system_of), 3)
    else:
        edges = (n_of.double() / 0.08) ** (1.0 / 3.0)
        points = _random(generator, len(system_of), 3)
        if case["system"] == "molecules":
            boxes = torch.zeros((n_systems, 3, 3), dtype=torch.float64, device="cuda")
            points = points * edges[system_of, None]
        else:
            shapes = torch.stack([_box_shape(skew) for skew in np.linspace(0.0, 0.4, 16)]).cuda()
            boxes = shapes[torch.randint(0, 16, (n_systems,), device="cuda", generator=generator)] * edges[:, None, None]
            points = (points[:, :, None] * boxes[system_of]).sum(dim=1)
    generator = _generator(seed)
    shuffled = torch.randperm(n_systems, device="cuda", generator=generator)
    place_of = torch.empty_like(shuffled)
    place_of[shuffled] = torch.arange(n_systems, device="cuda")
    points = points + _random(generator, n_systems, 3)[system_of]
    order = torch.argsort(place_of[system_of] + _random(generator, len(points)))
    first_point = np.concatenate([[0], np.cumsum(sizes[shuffled.cpu().numpy()])])
    return points[order].contiguous(), first_point, boxes[shuffled].contiguous(), case["system"] != "molecules"


def prepare(case, seed):
    """The calculator and its inputs, as a user's program holds them before the call."""
    state = dict(kind=case["kind"], quantities=case["quantities"], cutoff=case["cutoff"], sorted=case["sorted"])
    if case["kind"] == "batch":
        state["calculator"] = NeighborList(cutoff=case["cutoff"], full_list=case["full"], sorted=case["sorted"])
        state["batches"] = [_batch(case, number, 100 * seed + number) for number in range(case["batches"])]
        return state

    frames, box, periodic = _single_system(case, seed)
    if case["kind"] == "forces":
        from vesin_amd.torchscript import NeighborList as DifferentiableNeighborList

        state["calculator"] = DifferentiableNeighborList(cutoff=case["cutoff"], full_list=case["full"], sorted=case["sorted"])
        state["points"] = frames[0].requires_grad_()
        state["box"] = box.requires_grad_(case["box_gradient"])
        state["periodic"] = torch.tensor(periodic, device="cuda")
        return state

    state["calculator"] = NeighborList(
        cutoff=case["cutoff"], full_list=case["full"], sorted=case["sorted"], skin=case.get("skin", 0.0)
    )
    state["frames"], state["box"], state["periodic"] = frames, box, periodic
    if case["kind"] == "host":
        state["frames"], state["box"] = [frame.cpu().numpy() for frame in frames], box.cpu().numpy()
    return state


# ---- one pass


def run(state):
    calculator, quantities = state["calculator"], state["quantities"]
    if state["kind"] == "forces":
        return _forces(state)
    if state["kind"] == "batch":
        results = []
        for batch in state["batches"]:
            rows, first_pair = calculator.compute_batch(*batch, quantities)
            results.append((_indexable(rows), first_pair))
        return results
    return [_indexable(calculator.compute(frame, state["box"], state["periodic"], quantities)) for frame in state["frames"]]


def _indexable(outputs):
    """Pairs as the type that torch takes for indexing (a view)."""
    return [t.view(torch.int64) if isinstance(t, torch.Tensor) and t.dtype == torch.uint64 else t for t in outputs]


def _forces(state):
    """Gradients of a pair potential whose derivative is d - cutoff for the distances and a tenth of the vector for the
    vectors; the rows too where they come in an order of their own."""
    outputs = state["calculator"].compute(state["points"], state["box"], state["periodic"], state["quantities"])
    derivatives = []
    for letter, output in zip(state["quantities"], outputs):
        derivatives.append(output.detach() - state["cutoff"] if letter == "d" else output.detach() * 0.1)
    inputs = [state["points"]] + ([state["box"]] if state["box"].requires_grad else [])
    gradients = torch.autograd.grad(outputs, inputs, grad_outputs=derivatives)
    return gradients, [output.detach() for output in outputs] if state["sorted"] else None


# ---- what a pass cannot do without


def _rows(case):
    """About how many rows the list of a case has (of one batch or frame)."""
    sphere = 4.0 / 3.0 * math.pi * case["cutoff"] ** 3
    share = 1.0 if case["full"] else 0.5
    if case["system"] in ("diamond", "replicas"):
        points = 8 * case["replicas"] ** 3 * case.get("systems", 1)
        return share * points * (8 / DIAMOND_A**3 * sphere - 1)
    if case["system"] == "crystals":
        return share * _points(case) * 0.08 * sphere
    if case["system"] == "molecules":
        # points spread evenly in a cube: the share of pairs within the cutoff, by the closed form for short distances
        # and one beyond
        total = 0.0
        for n in range(case["smallest"], case["largest"] + 1):
            r = case["cutoff"] / (n / 0.08) ** (1.0 / 3.0)
            within = 1.0 if r >= 1.0 else math.pi * r**3 * (4 / 3 - 1.5 * r + 8 * r**2 / (5 * math.pi) - r**3 / (6 * math.pi))
            total += n * (n - 1) * min(1.0, within)
        return share * case["systems"] * total / (case["largest"] - case["smallest"] + 1)
    if case["system"] == "liquid":
        return share * case["points"] * case["density"] * sphere
    # pairs of one blob: distances of a Gaussian of sqrt(2) sigma; other blobs: their mean density in the volume of all
    x = case["cutoff"] / (8.0 * math.sqrt(2.0))
    within = math.erf(x / math.sqrt(2.0)) - math.sqrt(2.0 / math.pi) * x * math.exp(-(x**2) / 2)
    edge = 300.0 * (case["blobs"] / 50) ** (1.0 / 3.0)
    others = case["points"] * (case["blobs"] - 1) / case["blobs"] * min(1.0, sphere / edge**3)
    return share * case["points"] * (case["points"] / case["blobs"] * within + others)


def _points(case):
    if case["system"] in ("diamond", "replicas"):
        return 8 * case["replicas"] ** 3 * case.get("systems", 1)
    if "systems" in case:
        return case["systems"] * (case["smallest"] + case["largest"]) / 2
    return case["points"]


def work(case):
    """Every point read and every row written once (with a gradient: the rows' derivatives read once, the gradient
    written once), and the arithmetic of one distance per row."""
    value = 4 if case.get("dtype") == "float32" else 8
    rows, points = _rows(case), _points(case)
    if case["kind"] == "forces":
        per_row = {"d": value, "D": 3 * value}
        row_bytes = 2 * sum(per_row[letter] for letter in case["quantities"])
        return {"bytes": 2 * 3 * value * points + rows * row_bytes, "flops": 20 * rows}
    per_row = dict(BYTES_OF, d=value, D=3 * value, i=8, j=8)
    row_bytes = sum(per_row[letter] for letter in case["quantities"])
    passes = case.get("batches", 1) * case.get("frames", 1)
    return {"bytes": passes * (3 * value * points + rows * row_bytes), "flops": passes * 9 * rows}


def tolerance(case):
    """Rows are the same bit for bit. Gradients are sums in double precision whose order is not fixed (two runs differ by
    1e-14, and by 1e-13 where the terms of a point cancel most), rounded once to single precision where the caller's
    points are (6e-8 where a sum lies next to the middle of two numbers)."""
    if case["kind"] != "forces":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 2e-7, "max": 1e-6}
    return {"rel": 1e-13, "max": 1e-12}
