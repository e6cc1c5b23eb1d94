"""Which results of numpy callers come by way of pinned memory (vesin_amd/_host_results.py), without a GPU."""

import numpy as np
import pytest
import torch

from vesin_amd import _host_results
from vesin_amd._host_results import HostStaging

MB = 1_000_000
BYTES = {"i": 8, "j": 8, "P": 16, "S": 12, "d": 8, "D": 24}


# (quantities, bytes, time of a call through the pinned block over that of the copies one by one, whichever way through the
# block is the faster one)
@pytest.mark.parametrize("quantities, size, ratio", [
    ("d", 0.04 * MB, 1.07), ("d", 0.42 * MB, 1.08), ("d", 1.05 * MB, 1.04), ("d", 1.68 * MB, 0.89), ("d", 26.8 * MB, 0.53),
    ("PSdD", 0.31 * MB, 1.05), ("PSdD", 1.42 * MB, 1.06), ("PSdD", 1.88 * MB, 1.07), ("PSdD", 3.14 * MB, 0.90),
    ("PSdD", 50.3 * MB, 0.43), ("ijSd", 0.05 * MB, 0.77), ("ijSd", 0.85 * MB, 0.93), ("ijSd", 3.24 * MB, 0.88),
    ("ij", 0.18 * MB, 0.92), ("ij", 2.1 * MB, 0.87), ("ij", 53.6 * MB, 0.43), ("ij", 100 * MB, 1.0), ("PSdD", 100 * MB, 1.0),
])
def test_results_come_the_faster_way(quantities, size, ratio):
    rows = size / sum(BYTES[q] for q in quantities)
    sizes = [int(rows) * BYTES[q] for q in quantities]
    assert HostStaging().pays(sizes, columns="i" in quantities) == (ratio < 1.0)


@pytest.mark.parametrize("quantities", ["d", "D", "PS", "PSdD", "SSSSD", "i", "ijSd", "ijPSdD"])
def test_what_is_said_at_a_glance_is_what_the_sizes_say(quantities):
    staging, columns = HostStaging(), "i" in quantities
    said = set()
    for rows in [1, 2, 1000, *range(10_000, 60_000, 1000), *range(400_000, 9_000_000, 100_000)]:
        glance = staging.pays_at_a_glance(rows, len(quantities), columns)
        said.add(glance)
        assert glance is None or glance == staging.pays([rows * BYTES[q] for q in quantities], columns)
    assert said == {None, columns}


def test_no_rows_and_the_limit():
    staging = HostStaging()
    assert not staging.pays([0, 0], True)
    assert staging.pays([_host_results.LIMIT], False) and not staging.pays([_host_results.LIMIT + 1], False)


class _Event:
    def synchronize(self):
        pass


class _Stream(_Event):
    def record_event(self):
        return _Event()


@pytest.fixture
def no_gpu(monkeypatch):
    """Blocks of ordinary memory, copies that are done when they return."""
    empty = torch.empty

    def unpinned(*shape, pin_memory=False, device=None, **options):
        if pin_memory and torch.device(device or torch.get_default_device()).type != "cpu":
            raise RuntimeError("Only dense CPU tensors can be pinned")
        return empty(*shape, device=device, **options)

    monkeypatch.setattr(torch, "empty", unpinned)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _Stream())


def test_pinned_memory_that_is_refused(monkeypatch):
    """The results are copied one by one then, and the pool is as it was."""
    def refuse(*shape, **options):
        raise RuntimeError("out of memory")

    staging = HostStaging()
    monkeypatch.setattr(torch, "empty", refuse)
    assert staging.to_host([torch.arange(10)], [np.int64]) is None
    assert staging._held == 0 and staging._kept == []


@pytest.mark.parametrize("rows", [1000, 1_000_000])
def test_blocks_made_under_another_default_device(rows, no_gpu):
    values = torch.arange(rows, dtype=torch.float64)
    staging = HostStaging()
    with torch.device("meta"):
        assert np.array_equal(staging.to_host([values], [np.float64])[0], values.numpy())
    assert np.array_equal(staging.to_host([values], [np.float64])[0], values.numpy())
    assert staging._held > 0


def test_the_pool_never_locks_more_than_it_says(no_gpu, monkeypatch):
    """Counted at the allocator, which keeps pinned memory locked when a block is dropped."""
    locked = []
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda size, **options: locked.append(size) or empty(size, **options))
    staging = HostStaging()
    mb = 1 << 20
    # results of every size, growing and shrinking; several threads at once
    for sizes in [[k * mb] for k in (1, 2, 3, 9, 20, 40, 64, 30, 5)] + [[40 * mb, 40 * mb], [3 * mb] * 9, [64 * mb], [25 * mb] * 3]:
        blocks = [staging._take(size) for size in sizes]
        assert all(block is None or block.numel() >= size for block, size in zip(blocks, sizes))
        assert blocks[0] is not None  # (one thread always finds a block)
        for block in blocks:
            if block is not None:
                staging._give_back(block)
    assert sum(locked) == staging._held <= _host_results.POOL == 2 * _host_results.LIMIT
