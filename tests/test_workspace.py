"""The step's scratch buffers by name: views that are asked for again, buffers that grow."""
import pytest
import torch

from braidinfer_amd.engine.step import Workspace


@pytest.mark.parametrize("first, second", [((3, 4), (3, 4)), ((3, 4), (2, 4)), ((3, 4), (4, 3)), ((2, 3), (5, 7))])
def test_a_view_is_of_the_shape_asked_for_and_of_the_buffer_kept(first, second):
    ws = Workspace("cpu")
    a = ws.get("rows", first, torch.float32)
    b = ws.get("rows", list(second), torch.float32)
    assert tuple(a.shape) == first and tuple(b.shape) == second
    if b.numel() <= a.numel():
        assert a.data_ptr() == b.data_ptr()
    # back to the first shape: a view of the buffer kept now, not of one that growth replaced
    again = ws.get("rows", torch.Size(first), torch.float32)
    assert tuple(again.shape) == first and again.data_ptr() == b.data_ptr()
    assert ws.get("rows", second, torch.bfloat16).data_ptr() != b.data_ptr()
    ws.clear()
    c = ws.get("rows", second, torch.float32)
    assert tuple(c.shape) == second and c.dtype == torch.float32
