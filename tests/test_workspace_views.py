"""The views that the scratch buffers keep (CPU)."""

from __future__ import annotations

import weakref

import pytest
import torch

from dionw_amd import _workspace

CPU = torch.device("cpu")


@pytest.fixture(autouse=True)
def _clean():
    _workspace.release(CPU)
    yield
    _workspace.release(CPU)


def test_a_view_is_taken_again_only_where_it_fits() -> None:
    a = _workspace.buffer(CPU, "v", (4, 8), torch.float32, stream=1)
    assert _workspace.buffer(CPU, "v", (4, 8), torch.float32, stream=1) is a
    b = _workspace.buffer(CPU, "v", (8, 4), torch.float32, stream=1)
    assert b.shape == (8, 4) and b.data_ptr() == a.data_ptr()
    c = _workspace.buffer(CPU, "v", (4, 8), torch.int32, stream=1)
    assert c.dtype == torch.int32 and c.shape == (4, 8)
    assert _workspace.buffer(CPU, "v", (4, 8), torch.float32, stream=2).data_ptr() != a.data_ptr()


@pytest.mark.parametrize("how", ["release", "release_named", "regrow"])
def test_a_dropped_buffer_keeps_no_view(how: str) -> None:
    view = weakref.ref(_workspace.buffer(CPU, "v", (4,), torch.float32, stream=1))
    assert view() is not None  # held for the next request
    if how == "release":
        _workspace.release(CPU)
    elif how == "release_named":
        _workspace.release_named(CPU, 1, lambda name: name == "v")
    else:
        assert _workspace.buffer(CPU, "v", (1000,), torch.float32, stream=1).numel() == 1000
    assert view() is None
