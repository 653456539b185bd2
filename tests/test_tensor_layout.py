"""Block bookkeeping of ``BlockTensor`` on the CPU: sizes, default offsets, the
accepted forms of a block list, and the arrays that the C descriptor points to."""
import numpy as np
import pytest
import torch

from ultradmrg_amd.tensor import IN, OUT, Axis, BlockTensor

A = Axis.make([((0,), 3), ((1,), 1), ((2,), 4)], IN)
B = Axis.make([((0,), 2), ((1,), 5)], OUT)


@pytest.mark.parametrize("coords", [[], [(0, 0)], [(0, 0), (1, 1)], [[2, 1], [0, 0]],
                                    [tuple(np.int64(v) for v in c) for c in ((1, 0), (2, 1))],
                                    (c for c in ((0, 1), (2, 0)))], ids=["none", "one", "two", "lists", "numpy", "generator"])
def test_layout(coords):
    coords = list(coords) if not isinstance(coords, list) else coords
    sizes = [A.degs[a] * B.degs[b] for a, b in coords]
    t = BlockTensor([A, B], iter(coords), torch.zeros(max(sum(sizes), 1)))
    assert t.coords == [tuple(int(v) for v in c) for c in coords]
    assert all(type(v) is int for c in t.coords for v in c) and all(type(o) is int for o in t.offsets)
    assert t.offsets == [sum(sizes[:i]) for i in range(len(sizes))]
    assert t.size == sum(sizes)
    d = t.descriptor()
    assert d.nblocks == len(coords) and d.rank == 2
    assert [d.blk_coords[i] for i in range(2 * len(coords))] == [int(v) for c in coords for v in c]
    assert [d.blk_offset[i] for i in range(len(coords))] == t.offsets


def test_given_offsets_and_short_buffers():
    t = BlockTensor([A, B], [(0, 0), (2, 1)], torch.zeros(40), [20, 0])
    assert t.offsets == [20, 0] and t.size == 26
    with pytest.raises(ValueError):
        BlockTensor([A, B], [(0, 0), (2, 1)], torch.zeros(25), [20, 0])
    with pytest.raises(ValueError):
        BlockTensor._on_layout([A, B], [(0, 0)], [0], 6, torch.zeros(5))
    with pytest.raises(IndexError):
        BlockTensor([A, B], [(3, 0)], torch.zeros(40))


@pytest.mark.parametrize("offsets", [[20, 0], (20, 0), np.array([20, 0]), torch.tensor([20, 0]), iter([20, 0])],
                         ids=["list", "tuple", "array", "tensor", "iterator"])
def test_forms_of_offsets(offsets):
    t = BlockTensor([A, B], (iter(c) for c in ((0, 0), (2, 1))), torch.zeros(40), offsets)
    assert t.coords == [(0, 0), (2, 1)] and t.offsets == [20, 0] and t.size == 26


def test_uneven_coordinates_stay_as_given():
    t = BlockTensor([A, B], [(0, 1, 1), (0,)], torch.zeros(40))
    assert t.coords == [(0, 1, 1), (0,)] and t.offsets == [0, 15] and t.size == 18
