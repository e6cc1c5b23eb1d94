"""Results for callers that hold numpy arrays: the arrays of a call come to pinned host memory in one go, without a wait in
between, and from there to memory of their own, each while the next ones are still on the way. (They are not handed out where
they landed: pinned memory is not there for forked processes, and stays locked for as long as an array made of it lives.)

The pinned memory is kept in a pool of at most ``POOL`` bytes for the whole process, until it ends: blocks are never dropped, as
PyTorch's allocator would keep them locked. Results of more than ``LIMIT`` bytes, or that find no block, are copied one by one,
and so are those of a calculator's first call (it does not pay for the pinned memory).
"""

import threading

import numpy as np

LIMIT = 64 << 20      # bytes of results at most
POOL = 2 * LIMIT      # bytes of pinned memory, in use and kept: one block of every size, as blocks are powers of two
SMALLEST = 1 << 20    # bytes of a block at least
ALIGNMENT = 64        # of the arrays in a block
# Small results are waited for together, as an event for each array costs more than the overlap gives. That way through the
# block then only pays where it spares a copy of its own for the columns i and j. Up to 1 MB and three eighths of one per array
# (calls, copies one by one / together / each with an event, us: i j S d, 0.9 MB 220 / 204 / 234, 2.4 MB 316 / 300 / 291, 4.7 MB
# 429 / 417 / 345; P S d D, 0.7 MB 180 / 190 / 220, 2.5 MB 257 / 273 / 260, 3.1 MB 305 / 315 / 276; d, 0.2 MB 105 / 115 / 121, 1.1 MB
# 175 / 190 / 182, 1.7 MB 219 / 229 / 193; beyond, 8 to 50 MB, the last takes about half as long as the first)
SMALL = 1 << 20
SMALL_PER_ARRAY = 3 << 17


class HostStaging:
    def __init__(self):
        self._lock = threading.Lock()
        self._kept = []
        self._held = 0 # bytes of all blocks, none of which is ever dropped

    @staticmethod
    def _pinned(size):
        """A new block, or None when there is no pinned memory for it (a limit of the machine)."""
        import torch

        try:
            # (on the CPU, whatever torch's default device is)
            return torch.empty(size, dtype=torch.uint8, device="cpu", pin_memory=True)
        except RuntimeError:
            return None

    def _take(self, needed):
        with self._lock:
            fitting = [block for block in self._kept if block.numel() >= needed]
            if fitting:
                block = min(fitting, key=lambda b: b.numel())
                self._kept = [other for other in self._kept if other is not block]
                return block
            size = max(SMALLEST, 1 << (needed - 1).bit_length())
            if self._held + size > POOL:
                return None
            block = self._pinned(size)
            self._held += size if block is not None else 0
            return block

    def _give_back(self, block):
        with self._lock:
            self._kept.append(block)

    @staticmethod
    def _places(sizes):
        """Where arrays of these sizes start in a block, and where the last one ends."""
        starts, end = [], 0
        for size in sizes:
            starts.append(end)
            end += (size + ALIGNMENT - 1) // ALIGNMENT * ALIGNMENT
        return starts, end

    @staticmethod
    def _small(size, number):
        return size <= SMALL + number * SMALL_PER_ARRAY

    @classmethod
    def pays_at_a_glance(cls, rows, number, columns):
        """What `pays` says of `number` arrays of so many rows, of 24 bytes at most, whatever they are, or None (small calls
        take 100 us, of which adding up the sizes costs 2)."""
        size = (24 * rows + ALIGNMENT) * number
        if columns:
            return True if size <= LIMIT else None
        return False if cls._small(size, number) else None

    def fits(self, sizes):
        return 0 < self._places(sizes)[1] <= LIMIT

    def pays(self, sizes, columns):
        """Whether arrays of these sizes, some of them columns of the pairs or not, come faster this way than one by one."""
        return self.fits(sizes) and (columns or not self._small(self._places(sizes)[1], len(sizes)))

    def to_host(self, tensors, dtypes):
        """The device tensors (contiguous, of one device) as numpy arrays of the given types of the same size, or None when
        they do not fit."""
        import torch

        sizes = [tensor.numel() * tensor.element_size() for tensor in tensors]
        starts, needed = self._places(sizes)
        block = self._take(needed) if 0 < needed <= LIMIT else None
        if block is None:
            return None
        stream = torch.cuda.current_stream(tensors[0].device)
        in_one_go = self._small(needed, len(sizes))
        try:
            landing, landed = [], []
            for start, size, tensor in zip(starts, sizes, tensors):
                landing.append(block[start : start + size].view(tensor.dtype).view(tensor.shape))
                landing[-1].copy_(tensor, non_blocking=True)
                if not in_one_go:
                    landed.append(stream.record_event())
            if in_one_go:
                stream.synchronize()
                return [source.numpy().view(dtype).copy() for source, dtype in zip(landing, dtypes)]
            arrays = []
            for source, event, dtype in zip(landing, landed, dtypes):
                array = np.empty(tuple(source.shape), dtype=dtype)
                event.synchronize()
                # (torch's copy: by several threads where the array is large)
                torch.from_numpy(array.view(np.int64 if dtype == np.uint64 else dtype)).copy_(source)
                arrays.append(array)
            return arrays
        except BaseException:
            stream.synchronize() # (nothing is on its way into the block when it is given back)
            raise
        finally:
            self._give_back(block)


STAGING = HostStaging()
