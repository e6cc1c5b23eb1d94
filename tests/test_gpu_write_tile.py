"""sorted=True: the writing pass that gives every tile a workgroup (a list's second call on well-filled tiles) against the
oracle, bit for bit and in order."""

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
    "n,per_cell,skew,outside,periodic,used",
    [
        (70_000, 20.0, 0.3, 1, (True, True, True), "always"),
        (60_000, 18.5, 0.0, 0, (True, False, False), "always"),
        # enough points per tile without vectors, too few with
        (60_000, 19.0, 0.2, 0, (False, False, False), "without vectors"),  # (points outside would stretch the grid)
        (40_000, 11.0, 0.0, 1, (True, True, True), "without vectors"),
        (70_000, 27.0, 0.0, 0, (True, True, True), "never"),      # most tiles would have two chunks
    ],
)
def test_second_calls(n, per_cell, skew, outside, periodic, used, full, quantities, capfd, monkeypatch):
    points, box = _liquid(n, per_cell, 3.0, skew, outside, n + int(per_cell))
    _check(points, box, periodic, 3.0, full, quantities, used == "always" or (used == "without vectors" and "D" not in quantities),
           capfd, monkeypatch)


@pytest.mark.parametrize("quantities", ["PSd", "PSdD"])
@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("order", ["none", "cells"])
def test_tiles_of_two_chunks(order, full, quantities, capfd, monkeypatch):
    """653 candidates around a tile on average, more than the 704 of a chunk around some: their rows come from two chunks,
    of points in no order and of points numbered cell by cell (whose rows follow those of the point before)."""
    rng = np.random.default_rng(7)
    cutoff, side = 3.0, 14
    edge = 1.001 * cutoff * side
    points = edge * rng.random((int(24.2 * side**3), 3))
    if order == "cells":
        points = points[np.lexsort(np.floor(points / (edge / side)).T)]
    candidates = _check(points, edge * np.eye(3), (True, True, True), cutoff, full, quantities, True, capfd, monkeypatch)
    assert candidates > 704


def _check(points, box, periodic, cutoff, full, quantities, used, capfd, monkeypatch):
    """Three calls of one list against the oracle; `used`: whether the second and the third write by tiles. Returns the most
    candidates around a tile."""
    import torch

    expected = oracle.canonicalize(oracle.neighbors(points, box, list(periodic), cutoff, full, False, "ijSdD"))
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=cutoff, full_list=full, sorted=True)
    device_points, device_box = torch.tensor(points, device="cuda:0"), torch.tensor(box, device="cuda:0")
    for call in range(3):
        capfd.readouterr()
        outputs = calculator.compute(device_points, device_box, periodic, quantities)
        err = capfd.readouterr().err
        found = re.findall(r"most candidates of a tile (\d+), .* waves each( \(candidates in LDS\))? and counted by \d+: used", err)
        assert len(found) == 1, err
        assert (found[0][1] != "") == (used and call > 0), err
        for q, out in zip(quantities, outputs):
            assert np.array_equal(out.cpu().numpy(), expected[NAMES[q]]), (call, q)
    return int(found[0][0])
