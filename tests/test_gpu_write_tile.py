"""sorted=True: the writing pass that gives every tile a workgroup (from a list's second call on) against the oracle, bit for
bit and in order."""

import re

import numpy as np
import pytest

import oracle
from vesin_amd import NeighborList

pytestmark = pytest.mark.gpu

NAMES = {"P": "pairs", "S": "shifts", "d": "distances", "D": "vectors"}


def _liquid(n, per_cell, cutoff, skew, outside, seed):
    """`per_cell` points per cell of the search on average, of which some lie outside of the box."""
    rng = np.random.default_rng(seed)
    box = np.array([[1.0, 0.0, 0.0], [0.6 * skew, 1.05, 0.0], [skew, 0.4 * skew, 1.1]])
    box *= (n / per_cell) ** (1.0 / 3.0) * 1.04 * cutoff / np.linalg.det(box) ** (1.0 / 3.0)
    points = rng.random((n, 3))
    points[: n // 50] += outside * rng.integers(-2, 3, size=(n // 50, 3))
    return points @ box, box


@pytest.mark.parametrize("quantities", ["PSd", "PSdD", "P"])
@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize(
    "n,per_cell,skew,outside,periodic",
    [
        (70_000, 20.0, 0.3, 1, (True, True, True)),
        (60_000, 18.5, 0.0, 0, (True, False, False)),
        (60_000, 19.0, 0.2, 0, (False, False, False)),  # (points outside would stretch the grid)
        (40_000, 11.0, 0.0, 1, (True, True, True)),
        (70_000, 27.0, 0.0, 0, (True, True, True)),     # cells of more than 32 points: several tiles each
    ],
)
def test_second_calls(n, per_cell, skew, outside, periodic, full, quantities, capfd, monkeypatch):
    points, box = _liquid(n, per_cell, 3.0, skew, outside, n + int(per_cell))
    _check(points, box, periodic, 3.0, full, quantities, capfd, monkeypatch)


@pytest.mark.parametrize("quantities", ["PSd", "PSdD"])
@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("order", ["none", "cells"])
def test_tiles_of_two_chunks(order, full, quantities, capfd, monkeypatch):
    """37 points in every cell, more of them near its sides than inside, so 999 candidates around a tile, of which more than
    the 512 of a chunk have a hit: their rows come from two chunks, of points in no order and of points numbered cell by cell (whose rows follow those of the point
    before). In a half list that takes points of smaller indices than all around them: in no order those of every 27th cell,
    cell by cell those of the first."""
    rng = np.random.default_rng(7)
    cutoff, side = 3.0, 10
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), axis=-1).reshape(-1, 1, 3)
    points = 1.001 * cutoff * (grid + 0.001 + 0.998 * rng.beta(0.5, 0.5, (side**3, 37, 3))).reshape(-1, 3)
    if order == "none":
        first = (np.repeat(grid.reshape(-1, 3), 37, axis=0) % 3 == 0).all(axis=1)
        points = points[np.lexsort([rng.random(len(points)), ~first])]
    box = 1.001 * cutoff * side * np.eye(3)
    candidates, hits = _check(points, box, (True, True, True), cutoff, full, quantities, capfd, monkeypatch)
    assert candidates == 999 and hits > 512


def _check(points, box, periodic, cutoff, full, quantities, capfd, monkeypatch):
    """Three calls of one list against the oracle, the second and the third with a workgroup per tile. Returns the most
    candidates around a tile, and the most of them with a hit."""
    import torch

    expected = oracle.canonicalize(oracle.neighbors(points, box, list(periodic), cutoff, full, False, "ijSdD"))
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=cutoff, full_list=full, sorted=True)
    device_points, device_box = torch.tensor(points, device="cuda:0"), torch.tensor(box, device="cuda:0")
    for call in range(3):
        capfd.readouterr()
        outputs = calculator.compute(device_points, device_box, periodic, quantities)
        err = capfd.readouterr().err
        found = re.findall(
            r"most candidates of a tile (\d+), .* waves each( \(a workgroup per tile, (\d+) hits at most\))? and counted by \d+: used", err
        )
        assert len(found) == 1, err
        assert (found[0][1] != "") == (call > 0), err
        for q, out in zip(quantities, outputs):
            assert np.array_equal(out.cpu().numpy(), expected[NAMES[q]]), (call, q)
    return int(found[0][0]), int(found[0][2])
