"""Host: what the descriptors' C++ path leaves to the Python one, and the name pointers."""
import ctypes as C

import pytest
import torch

from mxopt import InvalidArg, _lib as L, optimizers as M


def test_nothing_but_device_tensors_and_none_is_described():
    a = M._arrs((None, None))
    assert [(x.data, x.n, x.dtype) for x in a] == [(None, 0, 0)] * 2
    for bad in (torch.zeros(3), torch.zeros(2, 2).to_sparse(), torch.zeros(3, dtype=torch.int64)):
        with pytest.raises(InvalidArg):
            M._arrs([None, bad])
    with pytest.raises(AttributeError):
        M._arrs([5])
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: x + len(M._arrs([x])))(torch.zeros(2, 3))


@pytest.mark.parametrize("names", [[], ["w"], ["model.layers.0.w", "é", ""], tuple("abc")])
def test_names(names):
    a = M._names(names)
    assert isinstance(a, C.Array) and list(a)[:len(names)] == [n.encode() for n in names]
    with pytest.raises((TypeError, AttributeError)):
        M._names([*names, 3])


def test_layout_of_a_descriptor():
    assert C.sizeof(L.Array) == 24 and (L.Array.data.offset, L.Array.n.offset, L.Array.dtype.offset) == (0, 8, 16)
