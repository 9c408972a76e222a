"""Layers of routed experts in a row: the rows normed by the experts' last launch against the next layer's norm on its own."""
from dataclasses import dataclass

import numpy as np
import pytest
import torch

import braidinfer_amd as B
from braidinfer_amd import StepEntry
from braidinfer_amd import kernels as K
from braidinfer_amd.config import LayerSpec, ModelSpec, PartSpec, ScheduleEntry, register_architecture, unregister_architecture
from braidinfer_amd.parts.feedforward import RoutedExperts

pytestmark = pytest.mark.gpu
W = 256


@dataclass
class ToyConfig:
    architecture: str = "ToyExpertsForCausalLM"
    norm: str = "rmsnorm"
    adds: bool = False
    vocab_size: int = 90
    hidden_size: int = W
    max_position_embeddings: int = 256

    @classmethod
    def from_dict(cls, d):
        return cls(**{k: v for k, v in d.items() if k in cls.__dataclass_fields__})

    def to_dict(self):
        return {"architectures": [self.architecture], **{k: getattr(self, k) for k in self.__dataclass_fields__}}


def toy_spec(cfg):
    rms = PartSpec("rmsnorm", {"size": W, "eps": 1e-5})
    second = PartSpec("rows", {"size": W}) if cfg.norm == "rows" else rms
    attn = PartSpec("gqa_attention", {"hidden_size": W, "num_heads": 4, "num_kv_heads": 2, "head_dim": 64, "window": None, "position": "rope"})
    experts = PartSpec("routed_experts", {"hidden_size": W, "intermediate_size": 128, "num_experts": 8, "top": 2})
    names = {"mixer": "attn.", "feed_forward": "moe.", "norm.mixer": "ln."}
    layers = [LayerSpec(f"t.{i}.", attn, experts, {"mixer": second if i == 1 else rms}, "parallel_residual", names) for i in range(3)]
    return ModelSpec(architecture=cfg.architecture, hidden_size=W, vocab_size=90, embedding=PartSpec("embedding", {"vocab_size": 90, "hidden_size": W}),
                     layers=layers, schedule=[ScheduleEntry(0, 0), ScheduleEntry(1, 1, adds_embedding=cfg.adds), ScheduleEntry(2, 2)], final_norm=rms,
                     lm_head=PartSpec("lm_head", {"vocab_size": 90, "hidden_size": W, "tied_to": None}),
                     positions={"rope": PartSpec("rope", {"rotary_dim": 64, "theta": 1e4, "pairing": "half"})}, max_position_embeddings=256,
                     embedding_prefix="t.embed.", final_norm_prefix="t.norm.", lm_head_prefix="t.head.")


def logits(cfg, dtype):
    engine = B.Engine.random(cfg, seed=4, dtype=dtype, max_tokens=512, max_seq_len=128, n_slots=3, std=0.08, vector_jitter=0.3)
    rng = np.random.default_rng(1)
    slots, out = [engine.alloc_slot() for _ in range(3)], []
    out.append(engine.step([StepEntry(s, rng.integers(0, 90, n).tolist(), [n - 1]) for s, n in zip(slots, (61, 20, 7))]))
    for _ in range(3):
        out.append(engine.step([StepEntry(s, [int(rng.integers(0, 90))], [0]) for s in slots]))
    return torch.cat(out)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("norm,adds,rides", [("rmsnorm", False, 2), ("rows", False, 1), ("rmsnorm", True, 1)])
def test_rows_handed_over(monkeypatch, norm, adds, rides, dtype):
    """The bits of both ways, prompts and single tokens; rows that are read without a norm, or that the embedding is added to
    first, are left to their own launch."""
    seen, combine = [], K.experts_combine

    def counted(*a, then=None, **how):
        seen.append(then is not None)
        return combine(*a, then=then, **how)
    register_architecture("ToyExpertsForCausalLM", ToyConfig, toy_spec)
    try:
        monkeypatch.setattr(K, "experts_combine", counted)
        got = logits(ToyConfig(norm=norm, adds=adds), dtype)
        if dtype == "bfloat16":
            assert seen[:3].count(True) == rides, seen[:3]
        monkeypatch.setattr(RoutedExperts, "norms_rows", False)
        del seen[:]
        want = logits(ToyConfig(norm=norm, adds=adds), dtype)
        assert not any(seen) and torch.equal(got, want) and torch.isfinite(want).all()
    finally:
        unregister_architecture("ToyExpertsForCausalLM")
