"""Routed experts that leave the rows normed for the layer that runs next: which norms they may apply, on the CPU with the
launches recorded."""
import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.config import PartSpec
from braidinfer_amd.parts import Runtime, build_part
from braidinfer_amd.parts.base import ResidualSink

CPU = torch.device("cpu")


class Buffers:
    def get(self, name, shape, dtype):
        return torch.empty(shape, dtype=dtype)


class Step:
    ws = Buffers()


def norm_of(kind, W):
    params = {"size": W} if kind in ("rows", "layer_scale", "dynamic_tanh") else {"size": W, "eps": 1e-5}
    part = build_part("norm", PartSpec(kind, params))
    part.load({t.name: torch.ones(t.shape) for t in part.weight_specs("n.")}, "n.", Runtime(CPU, torch.float32))
    return part


@pytest.mark.parametrize("kind,ahead", [("rmsnorm", True), ("layernorm", False), ("rows", False), ("layer_scale", False), ("dynamic_tanh", False)])
def test_the_norm_that_reads_the_rows_next(monkeypatch, kind, ahead):
    """An RMS norm rides on the sum of the experts' outputs; the norms that have no weight, another mean or another form do not."""
    W, T, top = 64, 3, 2
    calls = []
    monkeypatch.setattr(K, "experts_combine", lambda *a, **how: calls.append(how))
    part = build_part("feed_forward", PartSpec("routed_experts", {"hidden_size": W, "intermediate_size": 32, "num_experts": 4, "top": top}))
    part.rt = Runtime(CPU, torch.float32)
    x, h = torch.zeros(T, W), torch.zeros(T, W)
    sink = ResidualSink(x, norm_of(kind, W))
    part._join(torch.zeros(T * top, W), torch.zeros(T * top, dtype=torch.int32), torch.zeros(T, top), x, h, Step(), sink, store=False)
    assert len(calls) == 1 and ("then" in calls[0]) == ahead and (sink.prepared is not None) == ahead
