"""Batches of periodic systems whose grids are picked on the device (32 systems and more) against the same batches with
the grids picked on the host (VESIN_HIP_GRIDS=host): the same lists, the same errors, whatever the calls before were."""

import numpy as np
import pytest

from vesin_amd import NeighborList

pytestmark = pytest.mark.gpu


def _batch(n_systems, seed, smallest=1, largest=90, density=0.08, empty=False):
    rng = np.random.default_rng(seed)
    sizes = rng.integers(smallest, largest + 1, n_systems)
    if empty:
        sizes[rng.random(n_systems) < 0.2] = 0
    points, boxes = [], []
    for n in sizes:
        edge = (max(n, 1) / density) ** (1.0 / 3.0)
        box = edge * (np.diag([1.0, 1.1, 0.9]) + rng.uniform(-0.25, 0.25, size=(3, 3)))
        boxes.append(box)
        points.append(rng.uniform(-0.4, 1.4, size=(n, 3)) @ box)
    first_point = np.concatenate([[0], np.cumsum(sizes)])
    return np.concatenate(points).reshape(-1, 3), first_point, np.stack(boxes)


def _rows(calculator, batch, periodic=True, sort=False):
    import torch

    points, first_point, boxes = batch
    outputs, first_pair = calculator.compute_batch(
        torch.tensor(points, device="cuda:0"), first_point, torch.tensor(boxes, device="cuda:0"), periodic, "PSdD"
    )
    rows = [out.cpu().numpy() for out in outputs]
    if sort:
        system = np.repeat(np.arange(len(first_pair) - 1), np.diff(first_pair.astype(np.int64)))
        pairs, shifts = rows[0].astype(np.int64), rows[1]
        order = np.lexsort((shifts[:, 2], shifts[:, 1], shifts[:, 0], pairs[:, 1], pairs[:, 0], system))
        rows = [r[order] for r in rows]
    return rows + [first_pair]


def _rows_and_where(calculator, batch, capfd, periodic=True, sort=False):
    """The rows, and whether their grids were picked on the device."""
    capfd.readouterr()
    rows = _rows(calculator, batch, periodic, sort)
    return rows, "from grids picked on the device" in capfd.readouterr().err


def _same(one, other):
    for a, b in zip(one, other):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("full,sort", [(True, True), (False, True), (True, False), (False, False)])
@pytest.mark.parametrize("algorithm", ["auto", "cell_list", "brute_force"])
def test_lists(algorithm, full, sort, capfd, monkeypatch):
    """Other systems in every call, then the same ones again (which starts from the grids of the call before), then
    other boxes around as many points."""
    batches = [_batch(32, 1), _batch(300, 2, empty=True), _batch(1030, 3, 1, 12, 0.02)]
    batches += [batches[-1], (batches[-1][0], batches[-1][1], 1.05 * batches[-1][2]), _batch(31, 4), _batch(400, 5, 30, 200)]
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    results = {}
    for where in ("device", "host"):
        if where == "host":
            monkeypatch.setenv("VESIN_HIP_GRIDS", "host")
        calculator = NeighborList(cutoff=3.5, full_list=full, sorted=sort, algorithm=algorithm)
        results[where] = [_rows_and_where(calculator, batch, capfd, sort=not sort) for batch in batches]
    for (one, _), (other, _) in zip(results["device"], results["host"]):
        _same(one, other)
    # (not for the batch of the call before, nor for fewer than 32 systems)
    assert [picked for _, picked in results["device"]] == [True, True, True, False, True, False, True]
    assert not any(picked for _, picked in results["host"])


@pytest.mark.parametrize("sort", [True, False])
def test_a_single_system_in_between(sort):
    import torch

    batch = _batch(300, 7)
    calculator = NeighborList(cutoff=3.5, full_list=True, sorted=sort)
    expected = _rows(calculator, batch, sort=not sort)
    for _ in range(3):
        calculator.compute(torch.rand((500, 3), dtype=torch.float64, device="cuda:0") * 12.0,
                           torch.eye(3, dtype=torch.float64, device="cuda:0") * 12.0, True, "PSdD")
        for _ in range(2):
            _same(_rows(calculator, batch, sort=not sort), expected)


def test_open_directions_and_boxes_without_an_inverse(capfd, monkeypatch):
    """A batch with an open direction has its grids picked on the host, and so have the next 64 new ones."""
    import torch

    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    batch = _batch(300, 8)
    periodic = np.ones((300, 3), dtype=bool)
    periodic[17] = [True, False, True]
    periodic[18] = False
    on_host = NeighborList(cutoff=3.5, full_list=True, sorted=True)
    monkeypatch.setenv("VESIN_HIP_GRIDS", "host")
    expected, all_periodic = _rows(on_host, batch, torch.tensor(periodic)), _rows(on_host, batch)
    monkeypatch.delenv("VESIN_HIP_GRIDS")
    calculator = NeighborList(cutoff=3.5, full_list=True, sorted=True)
    _same(_rows(calculator, batch), all_periodic)
    for _ in range(2):
        for flags, right in ((torch.tensor(periodic), expected), (True, all_periodic)):
            rows, picked = _rows_and_where(calculator, batch, capfd, flags)
            _same(rows, right)
            assert not picked
    for bad, message in ((0.0, "not invertible"), (1e-3, "too large for this box")):
        calculator = NeighborList(cutoff=3.5, full_list=True, sorted=True)
        boxes = batch[2].copy()
        boxes[123] = bad * np.eye(3)
        with pytest.raises(RuntimeError, match=message):
            _rows(calculator, (batch[0], batch[1], boxes))
        _same(_rows(calculator, batch), all_periodic)


@pytest.mark.parametrize("n_systems", [32, 300])
def test_a_repeated_batch_sends_nothing_again(n_systems, capfd, monkeypatch):
    """What the sorted search needs of the division into systems goes to the device once for a batch that is called
    again, and again for another batch."""
    monkeypatch.setenv("VESIN_HIP_DEBUG", "1")
    calculator = NeighborList(cutoff=3.5, full_list=True, sorted=True)
    for batch in (_batch(n_systems, 9, 12), _batch(n_systems, 10, 12)):
        expected = _rows(NeighborList(cutoff=3.5, full_list=True, sorted=True), batch)
        sent = []
        for _ in range(4):
            capfd.readouterr()
            rows = _rows(calculator, batch)
            sent.append("first pairs of" in capfd.readouterr().err)
            _same(rows, expected)
        assert sent == [True, False, False, False]
