"""MixedStepBuffers.load on the CPU: the packed step, and what it refuses.

The device copy is a host copy here (no pinned memory, no event), so the packing
and the argument checks run without a GPU."""
import numpy as np
import pytest
import torch

from slo_attn.graph import MixedStepBuffers


class _Event:
    def synchronize(self):
        pass

    def record(self):
        pass


def _buffers(dc, pc, tc, width):
    b = object.__new__(MixedStepBuffers)
    b.dc, b.pc, b.tc, b.width = dc, pc, tc, width
    words = (dc + pc) * (2 + width)
    b._host = torch.zeros(8 * tc + 4 * words, dtype=torch.uint8)
    b._packed = torch.zeros_like(b._host)
    h = b._host.numpy()
    b._ids, b._words = h[:8 * tc].view(np.int64), h[8 * tc:].view(np.int32)
    b._copied = _Event()
    return b


def _loaded(b):
    p, rows = b._packed, b.dc + b.pc
    w = p[8 * b.tc:].view(torch.int32)
    return (p[:8 * b.tc].view(torch.int64).tolist(), w[:rows].tolist(), w[rows:2 * rows].tolist(),
            w[2 * rows:].view(rows, b.width).tolist())


def test_load_packs_the_step_and_clears_the_last_one():
    b = _buffers(3, 2, 12, 3)
    b.load([5, 900, 7], [(0, 4), (300, 5)], [[1], [2, 3, 4], [5], [6], [7, 8]], list(range(100, 112)))
    ids, start, tok, tab = _loaded(b)
    assert ids == list(range(100, 112)) and start == [5, 900, 7, 0, 300] and tok == [1, 1, 1, 4, 5]
    assert tab == [[1, -1, -1], [2, 3, 4], [5, -1, -1], [6, -1, -1], [7, 8, -1]]
    b.load([2], [(9, 2)], [[3], []], [40, 41, 42])
    ids, start, tok, tab = _loaded(b)
    assert ids == [40, 0, 0, 41, 42] + [0] * 7 and start == [2, 0, 0, 9, 0] and tok == [1, 0, 0, 2, 0]
    assert tab == [[3, -1, -1]] + [[-1] * 3] * 4


@pytest.mark.parametrize("ids", [[], [7], [7, 8]])
def test_load_refuses_fewer_ids_than_decode_rows(ids):
    b = _buffers(3, 1, 8, 2)
    with pytest.raises(IndexError):
        b.load([1, 2, 3], [], [[0], [1], [2]], ids)
    assert not b._packed.any()


def test_load_refuses_steps_that_do_not_fit():
    b = _buffers(2, 1, 6, 2)
    for args in (([1, 2, 3], [], [[0]] * 3, [1, 2, 3]), ([1], [(0, 6)], [[0], [1]], [1] * 7),
                 ([1], [], [], [1]), ([1], [], [[0, 1, 2]], [1])):
        with pytest.raises(ValueError):
            b.load(*args)
    with pytest.raises((ValueError, RuntimeError)):  # more ids than the step has room for
        b.load([1], [(0, 2)], [[0], [1]], [1] * 9)
