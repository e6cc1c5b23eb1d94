"""sorted=True: the writing pass that gives every tile a workgroup (a list's second call on well-filled tiles) against the
oracle, bit for bit and in order."""

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
        (70_000, 20.0, 0.3, 1, (True, True, True), True),     # some tiles have more than a chunk of candidates
        (60_000, 18.5, 0.0, 0, (True, False, False), True),
        (60_000, 19.0, 0.2, 0, (False, False, False), None),     # (points outside would stretch the grid: sparse cells)
        (40_000, 11.0, 0.0, 1, (True, True, True), None),     # enough points per tile without vectors, too few with
        (70_000, 27.0, 0.0, 0, (True, True, True), False),    # most tiles would have two chunks
    ],
)
def test_second_calls(n, per_cell, skew, outside, periodic, used, full, quantities, capfd, monkeypatch):
    import torch

    cutoff = 3.0
    points, box = _liquid(n, per_cell, cutoff, skew, outside, n + int(per_cell))
    expected = oracle.canonicalize(oracle.neighbors(points, box, list(periodic), cutoff, full, False, "ijSdD"))
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=cutoff, full_list=full, sorted=True)
    device_points, device_box = torch.tensor(points, device="cuda:0"), torch.tensor(box, device="cuda:0")
    for call in range(3):
        capfd.readouterr()
        outputs = calculator.compute(device_points, device_box, periodic, quantities)
        err = capfd.readouterr().err
        if call > 0 and used:
            assert "written by 4 waves each" in err, err
        for q, out in zip(quantities, outputs):
            assert np.array_equal(out.cpu().numpy(), expected[NAMES[q]]), (call, q)
