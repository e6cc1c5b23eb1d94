"""sorted=True on crowded cells: the in-order search without fixed sizes (forced with VESIN_HIP_SORT=crowded) gives the
list of the oracle, in the order (i, j, S), bit for bit; and the systems that the usual in-order search does not cover
come to it by themselves."""

import re

import numpy as np
import pytest

import oracle
from vesin_amd import NeighborList, configs

pytestmark = pytest.mark.gpu

NAMES = {"P": "pairs", "S": "shifts", "d": "distances", "D": "vectors"}


def _expected(points, box, periodic, cutoff, full):
    flags = [bool(periodic)] * 3 if isinstance(periodic, bool) else list(periodic)
    return oracle.canonicalize(oracle.neighbors(points, box, flags, cutoff, full, False, "ijSdD"))


def _compute(calculator, points, box, periodic, quantities="PSdD"):
    import torch

    outputs = calculator.compute(
        torch.tensor(np.ascontiguousarray(points), device="cuda:0"), torch.tensor(np.ascontiguousarray(box), device="cuda:0"),
        periodic, quantities,
    )
    return {NAMES[q]: out.cpu().numpy() for q, out in zip(quantities, outputs)}


def _check(points, box, periodic, cutoff, full, capfd, monkeypatch, covered=True, calls=2):
    expected = _expected(points, box, periodic, cutoff, full)
    monkeypatch.setenv("VESIN_HIP_SORT", "crowded")
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=cutoff, full_list=full, sorted=True)
    for call in range(calls):
        capfd.readouterr()
        result = _compute(calculator, points, box, periodic)
        lines = [line for line in capfd.readouterr().err.splitlines() if line.startswith("crowded search:")]
        # (after a system it does not cover, a list leaves that search alone for a while)
        assert len(lines) > 0 or (not covered and call > 0)
        assert result["pairs"].shape == expected["pairs"].shape
        for key in result:
            assert np.array_equal(result[key], expected[key]), (call, key)
    return int(re.search(r"(\d+) tiles in double precision", lines[-1]).group(1)) if lines else None


def _liquid(n, edge, seed, outside=0.0, skew=0.0):
    rng = np.random.default_rng(seed)
    box = edge * np.array([[1.0, 0.0, 0.0], [0.6 * skew, 1.05, 0.0], [skew, 0.4 * skew, 1.1]])
    return (rng.uniform(-outside, 1.0 + outside, size=(n, 3))) @ box, box


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("periodic", [(True, True, True), (True, False, True), (False, False, False)])
@pytest.mark.parametrize(
    "n,edge,cutoff,outside,skew",
    [
        (1, 5.0, 2.0, 0.0, 0.0),
        (33, 4.0, 3.0, 0.3, 0.2),       # one cell, a tile of 32 points would leave one over; images of the same points
        (700, 9.0, 3.0, 0.0, 0.3),      # 27 cells
        (2500, 12.0, 3.0, 0.6, 0.2),    # cells of 39 points (two tiles), points up to half a box outside
        (300, 30.0, 3.0, 0.0, 0.0),     # a third of a point per cell
        (4000, 9.0, 3.0, 0.0, 0.0),     # 148 points per cell, 4000 candidates: the sort of the most crowded cells
    ],
)
def test_liquids(n, edge, cutoff, outside, skew, periodic, full, capfd, monkeypatch):
    points, box = _liquid(n, edge, n, outside, skew)
    _check(points, box, periodic, cutoff, full, capfd, monkeypatch)


@pytest.mark.parametrize("n", [63, 64, 65, 255, 257, 767, 768, 769, 1535, 1537, 2047, 2048, 2049])
def test_numbers_of_candidates(n, capfd, monkeypatch):
    """One cell: n candidates for every point, around a unit, a chunk of the writing pass and the two sorts; most of
    them neighbours, more rows of a point than are lined up at a time."""
    rng = np.random.default_rng(n)
    _check(rng.random((n, 3)), np.eye(3), False, 1.3, n % 2 == 0, capfd, monkeypatch)


@pytest.mark.parametrize("n,covered", [(8192, True), (8193, False)])
def test_the_most_candidates(n, covered, capfd, monkeypatch):
    """27 cells in a periodic box: every point of the system is a candidate of every cell."""
    points, box = _liquid(n, 3.0, 5)
    _check(points, box, True, 0.999, False, capfd, monkeypatch, covered)


@pytest.mark.parametrize("order", ["lattice", "shuffled", "reversed"])
@pytest.mark.parametrize("full", [True, False])
def test_orders_of_the_points(order, full, capfd, monkeypatch):
    points, box, _ = configs.diamond(7, seed=3)
    if order == "shuffled":
        points = points[np.random.default_rng(1).permutation(len(points))]
    if order == "reversed":
        points = points[::-1]
    _check(points, box, True, 5.0, full, capfd, monkeypatch)


@pytest.mark.parametrize(
    "labels,n_dense",
    [
        ("a run and far ones", 1300), ("a run and far ones", 4500), ("runs near each other and a far one", 1300),
        ("runs near each other and a far one", 4500), ("powers", 1300), ("powers", 4500), ("images and far ones", 700),
    ],
)
def test_labels_that_clump(labels, n_dense, capfd, monkeypatch):
    """Original indices of a cell's candidates that are no even spread: nearly all in a small part of the range between
    the lowest and the highest, which is shared out again, once or several times; the order is the oracle's every time. The
    other points lie apart, on a lattice. In a long box, two cells wide, points come with their images."""
    rng = np.random.default_rng(n_dense)
    images = labels == "images and far ones"
    # (a bucket of the first sharing covers 98 indices or more; 68 in the long box, of which each comes twice on average)
    n, cutoff = 70_000 if images else 400_000, 3.0
    if labels in ("a run and far ones", "images and far ones"):
        dense = np.concatenate([np.arange(n_dense - 3), [n // 2, n - 2, n - 1]])
    elif labels == "powers":
        dense = np.unique(np.exp(np.linspace(0.0, np.log(n - 1.0), 4 * n_dense)).astype(int))
        dense = rng.permutation(dense)[:n_dense]
    else:
        dense = np.concatenate([np.arange(n_dense // 2), 5 + n_dense // 2 + np.arange(n_dense - n_dense // 2 - 1), [n - 1]])
    others = np.setdiff1d(np.arange(n), dense)
    side = 2 if images else int(np.ceil(len(others) ** (1 / 3)))
    grid = np.arange(len(others))
    lattice = 3.5 * np.stack([grid // side // side, grid // side % side, grid % side], axis=1)
    box = np.diag([15.0 + lattice[:, 0].max() + 5.0, *([7.0] * 2 if images else [15.0 + 3.5 * side + 5.0] * 2)])
    points = np.empty((n, 3))
    points[others] = lattice + ([15.0, 0.5, 0.5] if images else 15.0)
    points[dense] = np.array([8.9, 7.0, 7.0] if images else [8.9] * 3) * rng.random((len(dense), 3))
    _check(points, box, images, cutoff, False, capfd, monkeypatch)


def test_coincident_points_and_shifts_beyond_the_key(capfd, monkeypatch):
    points, box = _liquid(900, 9.0, 8)
    points[100:200] = points[0:100]
    _check(points, box, True, 3.0, True, capfd, monkeypatch)
    points[::2] += 300.0 * box[0]
    _check(points, box, True, 3.0, True, capfd, monkeypatch, covered=False)


def test_a_list_that_meets_other_systems(capfd, monkeypatch):
    """More points, more candidates around as many points, fewer rows: the room of the call before is too small, the
    arrays too."""
    monkeypatch.setenv("VESIN_HIP_SORT", "crowded")
    calculator = NeighborList(cutoff=3.0, full_list=True, sorted=True)
    # (2600 points: as many candidates around a cell of the smaller box, few in the larger one: the sort for the most
    # crowded cells has something to do in some calls and nothing in others)
    systems = [(500, 12.0), (2000, 12.0), (2000, 9.0), (2000, 20.0), (1000, 8.0), (1000, 8.0)]
    systems += [(2600, 20.0), (2600, 20.0), (2600, 9.0), (2600, 9.0), (2600, 20.0), (2600, 20.0)]
    for n, edge in systems:
        points, box = _liquid(n, edge, n)
        expected = _expected(points, box, True, 3.0, True)
        result = _compute(calculator, points, box, True)
        for key in result:
            assert np.array_equal(result[key], expected[key]), (n, edge, key)


@pytest.mark.parametrize("quantities", ["P", "PS", "Pd", "PD", "PSd"])
def test_quantities(quantities, monkeypatch):
    monkeypatch.setenv("VESIN_HIP_SORT", "crowded")
    points, box = _liquid(1200, 9.0, 4, 0.2, 0.2)
    expected = _expected(points, box, True, 3.0, False)
    calculator = NeighborList(cutoff=3.0, full_list=False, sorted=True)
    for _ in range(2):
        result = _compute(calculator, points, box, True, quantities)
        for key in result:
            assert np.array_equal(result[key], expected[key]), key


@pytest.mark.parametrize("kind", ["many candidates", "many rows", "blobs in a wide box", "sparse"])
def test_systems_that_come_by_themselves(kind, capfd, monkeypatch):
    """Called three times (first call, after the usual search reported that it does not cover the system, again), the
    last time in two halves. Systems of many, nearly empty tiles are counted once and left to the radix sort."""
    import torch

    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    rng = np.random.default_rng(2)
    if kind == "many candidates":
        (points, box), cutoff = _liquid(4000, 9.0, 1), 3.0
    elif kind == "many rows":
        points, box, cutoff = 1.5 * rng.random((600, 3)), 20.0 * np.eye(3), 3.0
    else:
        # boxes of 1.3 M cells: records of a fixed size per cell would take 2.4 GB and more
        box, cutoff = 220.0 * np.eye(3), 2.0
        if kind == "sparse":
            points = 220.0 * rng.random((200_000, 3))
        else:
            points = (220.0 * rng.random((50, 1, 3)) + 3.2 * rng.normal(size=(50, 4000, 3))).reshape(-1, 3)
    expected = _expected(points, box, True, cutoff, False)
    calculator = NeighborList(cutoff=cutoff, full_list=False, sorted=True)
    for call in range(3):
        capfd.readouterr()
        if call < 2:
            result = _compute(calculator, points, box, True)
        else:
            device_points, device_box = torch.tensor(points, device="cuda:0"), torch.tensor(box, device="cuda:0")
            calculator.enqueue(device_points, device_box, torch.tensor([True] * 3, device="cuda:0"), "PSdD")
            result = {NAMES[q]: out.cpu().numpy() for q, out in zip("PSdD", calculator.collect())}
        assert ("crowded search:" in capfd.readouterr().err) == (kind != "sparse" or call == 0)
        for key in result:
            assert np.array_equal(result[key], expected[key]), (call, key)


def test_the_rest_after_a_refused_system_ends(capfd, monkeypatch):
    """A list that met a system this search refuses leaves it alone for 64 calls, also where the usual in-order search is
    not tried either (records of a fixed size for so many cells would not fit), and takes it up again then."""
    import torch

    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    rng = np.random.default_rng(4)
    box, cutoff = 220.0 * np.eye(3), 2.0
    sparse = 220.0 * rng.random((200_000, 3))
    blobs = (220.0 * rng.random((50, 1, 3)) + 3.2 * rng.normal(size=(50, 4000, 3))).reshape(-1, 3)
    expected = _expected(blobs, box, True, cutoff, False)
    calculator = NeighborList(cutoff=cutoff, full_list=False, sorted=True)
    _compute(calculator, sparse, box, True)
    device_points, device_box = torch.tensor(blobs, device="cuda:0"), torch.tensor(box, device="cuda:0")
    tried = []
    for _ in range(66):
        capfd.readouterr()
        outputs = calculator.compute(device_points, device_box, True, "PSdD")
        err = capfd.readouterr().err
        assert "in-order search:" not in err
        tried.append("crowded search:" in err)
    assert tried == [False] * 64 + [True] * 2
    for q, out in zip("PSdD", outputs):
        assert np.array_equal(out.cpu().numpy(), expected[NAMES[q]]), q


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("periodic,far", [(False, 0.0), (False, 1.0e6), (True, 0.0), (True, 4.0e3)])
def test_pairs_next_to_the_cutoff(periodic, far, full, capfd, monkeypatch):
    """Pairs within a few units in the last place of the cutoff, on either side, which single precision cannot decide; far from
    the origin, and with points moved by box vectors, so that shifts and wraps take part in the decision."""
    rng = np.random.default_rng(9)
    cutoff, box = 3.0, np.array([[38.0, 0.0, 0.0], [4.0, 39.0, 0.0], [-3.0, 2.0, 40.0]])
    grid = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    first = (grid + 0.5 + rng.uniform(-0.05, 0.05, size=grid.shape)) / 12 @ box
    direction = rng.normal(size=first.shape)
    direction /= np.linalg.norm(direction, axis=1)[:, None]
    steps = rng.integers(-6, 7, size=len(first)).astype(np.float64)
    second = first + direction * (cutoff * (1.0 + steps * 2.0**-52))[:, None]
    points = np.concatenate([first, second])
    if periodic:
        points[::3] += rng.integers(-3, 4, size=points[::3].shape) @ box
    points = (points + far)[rng.permutation(len(points))]
    _check(points, box, periodic, cutoff, full, capfd, monkeypatch)
    expected = _expected(points, box, periodic, cutoff, full)
    assert (np.abs(expected["distances"] - cutoff) < 1e-8).sum() > 300
    assert not periodic or (expected["shifts"] != 0).any(axis=1).sum() > 300


@pytest.mark.parametrize("scale", [1e-6, 1e9, 1e12])
@pytest.mark.parametrize("full", [True, False])
def test_small_and_large_cutoffs(full, scale, capfd, monkeypatch):
    """The largest is left to double precision altogether (a square of 9e24); of points moved by box vectors too, and of tiles
    of which none was moved."""
    for outside in (0.0, 0.6):
        points, box = _liquid(4000, 20.0, 10, outside, 0.2)
        in_double = _check(points * scale, box * scale, True, 3.0 * scale, full, capfd, monkeypatch)
        assert (in_double > 0) == (scale == 1e12)


@pytest.mark.parametrize("full", [True, False])
def test_every_pair_in_double_precision(full, capfd, monkeypatch):
    """VESIN_HIP_TESTS=double."""
    points, box = _liquid(4000, 20.0, 10, 0.0, 0.2)
    moved = np.random.default_rng(16).integers(-2, 3, size=points.shape)
    moved[points[:, 0] < np.median(points[:, 0])] = 0
    assert _check(points + moved @ box, box, True, 3.0, full, capfd, monkeypatch) == 0
    monkeypatch.setenv("VESIN_HIP_TESTS", "double")
    assert _check(points + moved @ box, box, True, 3.0, full, capfd, monkeypatch) > 0


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("full", [True, False])
def test_tiles_too_wide_for_single_precision(full, periodic, capfd, monkeypatch):
    """Pairs of points in a box of 4,000 cutoffs, whose cells are 222 cutoffs wide (no more cells than points): the points of
    tiles with two pairs and more are too far apart for the tests in single precision, those of one pair are not."""
    rng = np.random.default_rng(14)
    first = 4000.0 * rng.random((1500, 3))
    points = np.concatenate([first, first + 0.6 * rng.normal(size=first.shape)])[rng.permutation(3000)]
    expected = _expected(points, 4000.0 * np.eye(3), periodic, 1.0, full)
    assert len(expected["pairs"]) > 500
    assert 0 < _check(points, 4000.0 * np.eye(3), periodic, 1.0, full, capfd, monkeypatch)


@pytest.mark.parametrize(
    "n,quantities,full,streamed",
    [
        (150_000, "P", True, True), (150_000, "PSd", True, True), (150_000, "PSdD", False, True),
        (100_000, "PSdD", False, False), # (by granule: see crowded_stores)
    ],
)
def test_lists_beyond_the_caches(n, quantities, full, streamed, capfd, monkeypatch):
    """More than 200 MB of rows: stored past the caches, with vectors only of systems whose shared pieces would not stay there."""
    points, box = _liquid(n, 3.03 * (n / 25.0) ** (1.0 / 3.0), 13, 0.0, 0.1)
    expected = _expected(points, box, True, 3.0, full)
    row_bytes = 16 + 12 * ("S" in quantities) + 8 * ("d" in quantities) + 24 * ("D" in quantities)
    assert len(expected["pairs"]) * row_bytes > 200 << 20 and len(expected["pairs"]) >= 40 * n
    assert streamed == ("D" not in quantities or n * 16 * row_bytes > 128 << 20)
    monkeypatch.setenv("VESIN_HIP_SORT", "crowded")
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=3.0, full_list=full, sorted=True)
    for call in range(2):
        capfd.readouterr()
        result = _compute(calculator, points, box, True, quantities)
        assert "crowded search:" in capfd.readouterr().err
        for key in result:
            assert np.array_equal(result[key], expected[key]), (call, key)
