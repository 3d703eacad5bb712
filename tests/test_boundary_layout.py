"""The copy of a boundary array into the kernels' layout is kept only while that
array lives unchanged: another one at its address gets a copy of its own."""
import numpy as np
import pytest
import torch


@pytest.fixture
def layout(monkeypatch):
    from pywrf_amd import _lib
    monkeypatch.setattr(_lib, "_require_device", lambda t: None)
    monkeypatch.setattr(_lib, "_bdy_copies", {})
    return _lib.boundary_layout


@pytest.mark.parametrize("kind,shape", [("x", (3, 7, 5)), ("y", (3, 5, 7))])
@pytest.mark.parametrize("view", [False, True])
def test_another_array_at_the_same_address(layout, kind, shape, view):
    storage = np.arange(105, dtype=np.float32)

    def array():
        t = torch.from_numpy(storage)
        return t.view(shape) if view else torch.from_numpy(storage.reshape(shape))
    a = array()
    assert torch.equal(layout(a, kind, 3, 7), a)
    del a
    storage += 1.0                     # the next owner of the memory, its version counter at 0 again
    b = array()
    assert torch.equal(layout(b, kind, 3, 7), b)


def test_one_array_is_copied_once_until_it_changes(layout):
    a = torch.rand(3, 7, 5)
    c = layout(a, "x", 3, 7)
    assert layout(a, "x", 3, 7) is c
    assert layout(a.view(3, 7, 5), "x", 3, 7) is c          # a view of it
    a.add_(1.0)
    d = layout(a, "x", 3, 7)
    assert d is not c and torch.equal(d, a)
    native = torch.rand(5, 3, 7).permute(1, 2, 0)
    assert layout(native, "x", 3, 7) is native
