"""Results of numpy callers by way of pinned memory (from a calculator's second call on): what the copies one by one give."""

import threading

import numpy as np
import pytest

from vesin_amd import NeighborList, _host_results, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("replicas", [1, 3, 5, 9])  # the last two: beyond what is waited for together
def test_later_calls_equal_the_first(replicas, dtype):
    points, box, _ = configs.diamond(replicas, seed=replicas)
    calculator = NeighborList(cutoff=5.0, full_list=True, sorted=True)
    first = calculator.compute(points.astype(dtype), box.astype(dtype), True, "ijPSdDi")
    kept = calculator.compute(points.astype(dtype), box.astype(dtype), True, "ijPSdDi")
    before = [array.copy() for array in kept]
    kept[0][:] = 7  # (every array has memory of its own)
    again = calculator.compute(points.astype(dtype), box.astype(dtype), True, "ijPSdDi")
    for a, b, c, k in zip(first, before, again, range(7)):
        assert a.dtype == b.dtype == c.dtype and c.flags.writeable and c.flags.c_contiguous
        assert np.array_equal(a, b) and np.array_equal(a, c), k
    assert all(np.array_equal(a, b) for a, b in zip(kept[1:], before[1:]))


def test_beyond_the_limit_and_without_rows(monkeypatch):
    points, box, _ = configs.diamond(4, seed=1)
    calculator = NeighborList(cutoff=5.0, full_list=True, sorted=True)
    first = calculator.compute(points, box, True, "ijSd")
    monkeypatch.setattr(_host_results, "LIMIT", 1000)
    assert all(np.array_equal(a, b) for a, b in zip(first, calculator.compute(points, box, True, "ijSd")))
    monkeypatch.undo()
    nothing = NeighborList(cutoff=0.1, full_list=True)
    for _ in range(3):
        i, S, d = nothing.compute(points, box, True, "iSd")
        assert i.shape == (0,) and S.shape == (0, 3) and d.shape == (0,)


@pytest.mark.parametrize("quantities", ["ij", "jd", "PSdDi"])
def test_nothing_is_made_for_results_that_do_not_fit(quantities, monkeypatch):
    """Results beyond the limit take no more device memory than the copies one by one do."""
    import torch

    points, box, _ = configs.diamond(12, seed=2)

    def peak_and_results(limit):
        monkeypatch.setattr(_host_results, "LIMIT", limit)
        calculator = NeighborList(cutoff=5.0, full_list=True, sorted=True)
        for _ in range(3):
            torch.cuda.reset_peak_memory_stats()
            results = calculator.compute(points, box, True, quantities)
        return torch.cuda.max_memory_allocated(), results

    monkeypatch.setattr(NeighborList, "_host_results", lambda self, *arguments: None)
    one_by_one, expected = peak_and_results(0)
    monkeypatch.undo()
    beyond, results = peak_and_results(1000)
    assert beyond <= one_by_one
    assert all(np.array_equal(a, b) for a, b in zip(expected, results))


def test_several_threads():
    systems = [configs.diamond(replicas, seed=replicas)[:2] for replicas in (2, 3, 4, 5)]
    expected = [NeighborList(cutoff=5.0, full_list=True, sorted=True).compute(p, b, True, "PSd") for p, b in systems]
    failures = []

    def work(k):
        calculator = NeighborList(cutoff=5.0, full_list=True, sorted=True)
        for _ in range(8):
            results = calculator.compute(*systems[k], True, "PSd")
            if not all(np.array_equal(a, b) for a, b in zip(results, expected[k])):
                failures.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert failures == []
