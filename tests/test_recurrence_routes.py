"""Which kernel walks a step's sequences through the recurrences, by their numbers of tokens: the rule alone, on the host."""
import itertools

import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.parts import delta_rule, gated_recurrence, time_mix
from braidinfer_amd.parts.base import MixerContext

FROM = gated_recurrence.CHUNKS_FROM


class Workspaces:
    def get(self, name, shape, dtype):
        return torch.empty(shape, dtype=dtype, device="meta")


class Step:
    def __init__(self, lens):
        self.host_new, self.n_seqs, self.n_tokens, self.max_new = list(lens), len(lens), sum(lens), max(lens)
        self.host_slots, self.is_decode, self.ws, self.extras = list(range(len(lens))), all(n == 1 for n in lens), Workspaces(), {}
        self.tokens = self.cu_seqlens = self.slots = self.seq_of_token = torch.zeros(1, dtype=torch.int32)
        self.position_data = {}


def mixer(kind, d, heads):
    if kind == "hgrn2":
        part = gated_recurrence.HGRN2(64, heads, d, 32, 1e-5)
    elif kind == "wkv":
        part = time_mix.WKVTimeMix(64, heads, d, 8, 1e-5)
        part.w = {s: None for s in ("r", "k", "v", "g", "w1", "w2")}
    elif kind == "delta":
        part = delta_rule.GatedDeltaRule(64, heads, heads, d, 32, 4, 1e-5)
        part.conv = part.conv_t = None
    else:
        part = delta_rule.LightningAttention(64, heads, d, 32, [0.9] * heads, 1e-5)
    part.rt = type("Runtime", (), {"dtype": torch.float32})
    return part


def walks(monkeypatch, kind, lens, d=64, heads=64):
    """For every sequence the kernels that walk it, from the arguments of the launches."""
    by = [[] for _ in lens]

    def scan(name):
        def launch(*a, below=0, least=0, singles=None, **k):
            mine = [i for i, n in enumerate(lens) if n >= least and not (below and n >= below)]
            assert mine, "a launch that walks nothing"
            if singles is not None:
                assert singles == all(lens[i] <= 1 for i in mine)
            for i in mine:
                by[i].append(name)
        return launch
    for name in ("chunk_scan", "glr_scan", "glr_scan_pieces", "wkv_scan", "wkv_scan_pieces", "dr_scan", "dr_scan_pieces"):
        monkeypatch.setattr(K, name, scan("chunks" if name == "chunk_scan" else "pieces" if name.endswith("pieces") else "walk"))
    for name in ("shift_mix", "tanh", "dr_conv_prepare", "head_rmsnorm", "head_norm_gate", "silu_rows"):
        monkeypatch.setattr(K, name, lambda *a, **k: None)
    monkeypatch.setattr(K, "device_cus", lambda: 256)
    monkeypatch.setattr(K, "glr_rows_per_lane", lambda d: 4 if d <= 64 else 8)
    for module in (delta_rule, gated_recurrence, time_mix):
        monkeypatch.setattr(module, "linear", lambda *a, **k: None)
    part = mixer(kind, d, heads)
    need = part.state_need()
    state = torch.empty((len(lens),) + tuple(need.shape), device="meta")
    part.forward(torch.empty(sum(lens), 64, device="meta"), torch.empty(sum(lens), 64, device="meta"), Step(lens), MixerContext(state=state))
    assert all(len(b) == 1 for b in by), by
    return [b[0] for b in by]


@pytest.mark.parametrize("kind", ["hgrn2", "wkv", "delta", "lightning"])
def test_every_sequence_by_its_own_tokens(monkeypatch, kind):
    for lens in ((1,) * 5, (FROM,), (FROM - 1,), (FROM,) + (1,) * 63, (1, 5000, 1), (FROM, FROM - 1, 300, 7, 1), (2, 40, FROM - 1), (500, 96, 128)):
        got = walks(monkeypatch, kind, lens)
        assert got == ["chunks" if n >= FROM else "walk" for n in lens], lens


@pytest.mark.parametrize("kind", ["hgrn2", "wkv", "delta", "lightning"])
def test_heads_that_chunks_do_not_take(monkeypatch, kind):
    assert set(itertools.chain(*(walks(monkeypatch, kind, lens, d=48) for lens in ((1, 1), (200, 1), (400,))))) == {"walk"}
    assert walks(monkeypatch, kind, (2000, 1), d=48, heads=16) == ["walk" if kind == "delta" else "pieces"] * 2


@pytest.mark.parametrize("kind", ["hgrn2", "wkv", "delta", "lightning"])
def test_lone_prompts_through_few_heads(monkeypatch, kind):
    # columns of 16 to a head: 2, WKV 4; 1,024 workgroups fill the chip, a piece has 128 tokens at least
    per_head = 4 if kind == "wkv" else 2
    for heads, tokens, pieces in ((2, 8192, 16), (1024 // per_head // 12, 8192, 12), (1024 // per_head // 11, 8192, 11), (2, 12 * 128, 12),
                                  (2, 12 * 128 - 1, 11), (2, 600, 4), (1024 // per_head // 8, 8192, 8)):
        got = walks(monkeypatch, kind, (tokens,), heads=heads)
        assert got == ["pieces" if pieces >= 12 and kind != "delta" else "chunks"], (heads, tokens)


@pytest.mark.parametrize("delta", [False, True])
def test_scratch_of_long_steps_is_bounded(monkeypatch, delta):
    H, d, e = 32, 128, 128
    block = K.chunk_block_floats(H, d, e, delta)
    for lens, floats in (((2048, 1), K.chunk_scratch_floats(2049, 2, H, d, e, delta)), ((200000, 1, 1), gated_recurrence.CHUNK_SCRATCH // 4),
                         ((FROM,) * 2000, 2000 * block)):
        a = gated_recurrence.chunk_scratch(Step(lens), H, d, e, delta)
        assert a["scratch"].numel() == floats and a["least"] == FROM and a["longs"] == sum(n >= FROM for n in lens)
        assert floats >= a["longs"] * block
