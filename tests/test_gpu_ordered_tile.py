"""sorted=True from a list's second call on: the search that gives every tile a workgroup, against the oracle, bit for bit and
in order, at the sizes where its pieces end (units, lines, chunks, windows of indices, ways to store)."""

import re

import numpy as np
import pytest

import oracle
from vesin_amd import NeighborList

pytestmark = pytest.mark.gpu

NAMES = {"P": "pairs", "S": "shifts", "d": "distances", "D": "vectors"}
EVERY = (True, True, True)


def _check(points, box, periodic, cutoff, full, quantities, capfd, monkeypatch):
    import torch

    expected = oracle.canonicalize(oracle.neighbors(points, box, list(periodic), cutoff, full, False, "ijSdD"))
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    monkeypatch.setenv("VESIN_HIP_LAUNCHES", "separate")  # (small systems: not in one launch)
    calculator = NeighborList(cutoff=cutoff, full_list=full, sorted=True)
    device_points, device_box = torch.tensor(points, device="cuda:0"), torch.tensor(box, device="cuda:0")
    for call in range(3):
        capfd.readouterr()
        outputs = calculator.compute(device_points, device_box, periodic, quantities)
        err = capfd.readouterr().err
        found = re.findall(r"tiles written by \d+ waves each(.*) and counted by \d+: used", err)
        assert len(found) == 1, err
        assert ("a workgroup per tile" in found[0]) == (call > 0), err
        for q, out in zip(quantities, outputs):
            assert np.array_equal(out.cpu().numpy(), expected[NAMES[q]]), (call, q)
    return expected, err


def _tiles(err):
    return int(re.search(r"(\d+) tiles written by", err).group(1))


def _in_double(err):
    return int(re.search(r"of (\d+) by a workgroup in double precision", err).group(1))


def _liquid(n, per_cell, cutoff, skew, seed):
    rng = np.random.default_rng(seed)
    box = np.array([[1.0, 0.0, 0.0], [0.6 * skew, 1.05, 0.0], [skew, 0.4 * skew, 1.1]])
    box *= (n / per_cell) ** (1.0 / 3.0) * 1.04 * cutoff / np.linalg.det(box) ** (1.0 / 3.0)
    return rng.random((n, 3)) @ box, box


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("quantities", ["PSd", "PSdD"])
@pytest.mark.parametrize(
    "n,per_cell",
    [
        (3_000, 2.0),    # tiles of a point or two, a unit of candidates
        (3_001, 4.7),    # two units: half of the waves have none
        (6_000, 9.4),    # four units
        (9_000, 14.2),   # six units, up to two per wave
        (9_000, 21.0),   # ten units and more
        (7_003, 26.0),   # up to sixteen units, cells of more than 32 points: several tiles each
        (70_000, 11.0),  # more indices than one round of the bit set
    ],
)
def test_fillings(n, per_cell, quantities, full, capfd, monkeypatch):
    points, box = _liquid(n, per_cell, 3.0, 0.2, n + int(per_cell))
    _check(points, box, EVERY, 3.0, full, quantities, capfd, monkeypatch)


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("periodic", [EVERY, (True, False, True), (False, False, False)])
def test_points_moved_by_box_vectors_and_open_directions(periodic, full, capfd, monkeypatch):
    points, box = _liquid(8_000, 12.0, 3.0, 0.3, 5)
    rng = np.random.default_rng(6)
    moved = np.zeros((8_000, 3))
    moved[::3] = rng.integers(-2, 3, size=moved[::3].shape)
    points = points + (moved * np.array(periodic)) @ box
    _check(points, box, periodic, 3.0, full, "PSdD", capfd, monkeypatch)


@pytest.mark.parametrize("full", [True, False])
def test_boxes_whose_stencil_sees_a_point_twice(full, capfd, monkeypatch):
    """Two cells along one direction: the candidates of a tile hold two images of the same points."""
    rng = np.random.default_rng(8)
    box = np.diag([6.4, 31.0, 31.0])
    _check(rng.random((4_000, 3)) @ box, box, EVERY, 3.0, full, "PSd", capfd, monkeypatch)


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("far", [0.0, 1.0e6])
def test_pairs_next_to_the_cutoff(far, full, capfd, monkeypatch):
    """Pairs within a few units in the last place of the cutoff, on either side, which single precision cannot decide; far
    from the origin too, where double precision itself leaves 1e-10 in a coordinate."""
    rng = np.random.default_rng(9)
    cutoff, box = 3.0, np.eye(3) * 38.0
    grid = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    first = (grid + 0.5 + rng.uniform(-0.05, 0.05, size=grid.shape)) / 12 @ box
    direction = rng.normal(size=first.shape)
    direction /= np.linalg.norm(direction, axis=1)[:, None]
    steps = rng.integers(-6, 7, size=len(first)).astype(np.float64)
    second = first + direction * (cutoff * (1.0 + steps * 2.0**-52))[:, None]
    points = np.concatenate([first, second]) + far
    expected, _ = _check(points, box, (False, False, False), cutoff, full, "PSd", capfd, monkeypatch)
    assert (np.abs(expected["distances"] - cutoff) < 1e-9).sum() > 300


@pytest.mark.parametrize("scale", [1e-6, 1e9, 1e12])
def test_small_and_large_cutoffs(scale, capfd, monkeypatch):
    """The largest is left to double precision altogether (a square of 9e24)."""
    points, box = _liquid(4_000, 12.0, 3.0, 0.2, 10)
    _, err = _check(points * scale, box * scale, EVERY, 3.0 * scale, True, "PSdD", capfd, monkeypatch)
    assert _in_double(err) == (_tiles(err) if scale == 1e12 else 0)


@pytest.mark.parametrize("full", [True, False])
def test_every_pair_in_double_precision(full, capfd, monkeypatch):
    """VESIN_HIP_TESTS=double, on points of which some were moved by box vectors, and others are in tiles of none that was."""
    points, box = _liquid(8_000, 12.0, 3.0, 0.3, 15)
    moved = np.random.default_rng(16).integers(-2, 3, size=points.shape)
    moved[points[:, 0] < np.median(points[:, 0])] = 0
    _, err = _check(points + moved @ box, box, EVERY, 3.0, full, "PSdD", capfd, monkeypatch)
    assert _in_double(err) == 0
    monkeypatch.setenv("VESIN_HIP_TESTS", "double")
    _, err = _check(points + moved @ box, box, EVERY, 3.0, full, "PSdD", capfd, monkeypatch)
    assert _in_double(err) == _tiles(err) > 0


def test_more_rows_than_a_line_holds(capfd, monkeypatch):
    """A blob of 37 points in every cell, about 150 rows for each of the 32 points of its first tile, where a line holds 2,560
    rows: two lines, of points in order of the cells (runs of many rows) and in none."""
    rng = np.random.default_rng(11)
    edge = 4 * 3.003
    centres = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * 3.003 + 1.5
    ball = np.clip(rng.normal(size=(64, 37, 3)) * 0.35, -1.4, 1.4)
    points = (centres[:, None, :] + ball).reshape(-1, 3)
    box = np.eye(3) * edge
    for order in (np.arange(len(points)), rng.permutation(len(points))):
        expected, _ = _check(points[order], box, EVERY, 3.0, True, "PSdD", capfd, monkeypatch)
        rows = np.empty(len(points), dtype=int)
        rows[order] = np.bincount(expected["pairs"][:, 0].astype(int), minlength=len(points))
        assert np.sort(rows.reshape(64, 37), axis=1)[:, :32].sum(axis=1).min() > 2560 and rows.max() <= 256


def _spans_of_cells(pairs, points, shape, n):
    """Of the neighbours of the points of every cell of the search: the range of their indices, as it is and counted from the
    last index on to the first where that is shorter."""
    cells = np.floor(points / (np.array(shape) * 3.567) * np.floor(np.array(shape) * 3.567 / 5.0)).astype(int)
    _, cell = np.unique(cells, axis=0, return_inverse=True)
    cell = cell.reshape(-1)
    first = np.full(cell.max() + 1, n)
    np.minimum.at(first, cell, np.arange(n))
    i, j = pairs.astype(np.int64).T
    ranges = []
    for index in (j, (j - first[cell[i]] + n // 2) % n):
        low, high = np.full(len(first), n), np.full(len(first), -1)
        np.minimum.at(low, cell[i], index)
        np.maximum.at(high, cell[i], index)
        ranges.append(high - low + 1)
    return ranges[0], np.minimum(*ranges)


@pytest.mark.parametrize("order", ["lattice", "none", "around the end"])
def test_orders_of_the_indices(order, capfd, monkeypatch):
    """Ranked through the bit set (65,536 indices at a time: one round, two, from the last index on to the first) or through
    buckets."""
    basis = np.array([[0, 0, 0], [0, 2, 2], [2, 0, 2], [2, 2, 0], [1, 1, 1], [1, 3, 3], [3, 1, 3], [3, 3, 1]]) / 4.0
    shape = (8, 46, 46) if order == "around the end" else (27, 27, 27)
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in shape], indexing="ij"), axis=-1).reshape(-1, 3)
    points = (cells[:, None, :] + basis[None, :, :]).reshape(-1, 3) * 3.567
    rng = np.random.default_rng(12)
    points += rng.normal(scale=0.05, size=points.shape)
    if order == "none":
        points = points[rng.permutation(len(points))]
    expected, err = _check(points, np.diag(np.array(shape) * 3.567), EVERY, 5.0, True, "PSd", capfd, monkeypatch)
    windowed, bucketed = (int(k) for k in re.search(r"candidates of (\d+) tiles ordered by window and of (\d+) by buckets", err).groups())
    as_it_is, around = _spans_of_cells(expected["pairs"], points, shape, len(points))
    if order == "none":
        assert windowed == 0 and bucketed > 4096 and around.min() > 2 * 65_536
    else:
        # (most of the cells, as the points on their edges may be in the next one)
        assert windowed > 4096 and bucketed == 0
        assert np.mean(around < 65_536) > 0.99 if order == "lattice" else np.mean((around > 65_536) & (around < 2 * 65_536)) > 0.5
        assert np.sum(as_it_is > 2 * 65_536) > 100


@pytest.mark.parametrize("quantities,full", [("P", True), ("PSd", True), ("PSdD", False)])
def test_lists_beyond_the_caches(quantities, full, capfd, monkeypatch):
    """More than 200 MB of rows: stored past the caches, all of them (pairs alone) or but for the ends of the runs."""
    points, box = _liquid(150_000, 25.0, 3.0, 0.1, 13)
    expected, _ = _check(points, box, EVERY, 3.0, full, quantities, capfd, monkeypatch)
    row_bytes = 16 + 12 * ("S" in quantities) + 8 * ("d" in quantities) + 24 * ("D" in quantities)
    assert len(expected["pairs"]) * row_bytes > 200 << 20
