"""Which products a step of routed experts goes through, by its tokens and widths: the rule alone, on the host."""
import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.parts import feedforward


class Workspaces:
    """Buffers without memory, but for what the host reads."""

    def get(self, name, shape, dtype):
        return torch.zeros(shape, dtype=dtype) if name == "moe_first" else torch.empty(shape, dtype=dtype, device="meta")


class Step:
    def __init__(self, tokens, is_decode):
        self.n_tokens, self.is_decode, self.ws = tokens, is_decode, Workspaces()


def route(monkeypatch, tokens, decode=False, W=4096, F=1792, E=32, top=8, dtype=torch.bfloat16):
    """The experts' launches of a step, in order."""
    called = []
    for name in ("route_topk", "experts_sort", "experts_up", "experts_down", "experts_up_grouped", "experts_down_grouped",
                 "experts_up_tiles", "experts_gather", "experts_gemm", "experts_combine", "silu_mul", "gemm"):
        monkeypatch.setattr(K, name, lambda *a, _name=name, **k: called.append(_name))
    monkeypatch.setattr(feedforward, "linear", lambda *a, **k: None)
    part = feedforward.RoutedExperts(W, F, E, top)
    part.rt, part.n_scores = type("Runtime", (), {"dtype": dtype}), E
    part.w_gu = part.w_down = [torch.empty(0)] * E
    part.forward(torch.empty((tokens, W), dtype=dtype, device="meta"), torch.empty((tokens, W), device="meta"), Step(tokens, decode))
    return [n for n in called if n not in ("route_topk", "experts_sort", "experts_combine")]


TILES = ["experts_up_tiles", "experts_gemm"]


# 149,796 tokens of 8 x 1,792: the last whose rows of the second product lie below 4 GB; 524,287 of 4,096: whose inputs do
@pytest.mark.parametrize("tokens,want", [(1801, TILES), (149796, TILES), (149797, TILES), (524287, TILES), (524288, ["experts_gather"]),
                                         (700000, ["experts_gather"])])
def test_steps_of_very_many_tokens(monkeypatch, tokens, want):
    # beyond: the rows gathered, and (from 1,536 pairs an expert) the products expert by expert, none of which the empty lists hold
    assert route(monkeypatch, tokens) == want


@pytest.mark.parametrize("W,F", [(4096, 1792), (2048, 1408), (64, 64)])
def test_tiles_say_what_they_take(W, F):
    last = (2 ** 32 - 1) // (2 * W)
    assert K.experts_tiles_take(torch.bfloat16, W, F, last) and not K.experts_tiles_take(torch.bfloat16, W, F, last + 1)
    assert not K.experts_tiles_take(torch.float32, W, F, 100)
    for w, f in ((W + 8, F), (W, F + 8), (2 ** 17, 2 ** 14), (2 ** 14, 2 ** 17)):          # matrices of 4 GB an expert
        assert not K.experts_tiles_take(torch.bfloat16, w, f, 100)
