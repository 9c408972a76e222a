"""HGRN2: linear attention whose forget gate also decides what is written.

Per token and head (d query channels, e value channels): q = silu(W_q n), v = W_v n,
f = lower + (1 - lower) * sigmoid(W_f n + b) per channel with a learnt lower bound, then
    S_t = diag(f_t) S_(t-1) + (1 - f_t) v_t^T,     o_t = S_t^T q_t
(the gate acts on the rows of S that belong to q's channels; no key, no other scale).  Every
head's o is RMS-normed over its e channels with one weight shared by the heads, the heads are
concatenated and projected by W_o.

The state S [heads, d, e] starts at zero, lives in float in both precisions and is carried from
step to step in the sequence's slot of the cache's state area (`StateNeed`, laid out as the scan
kernel's lanes hold it); the gates' activations, the recurrence and the head norm are float.
Prompts are walked token by token inside one kernel, a workgroup per 16 columns of a head's state
with the state in registers and the tokens' rows staged through LDS a chunk ahead; prompts through heads of 64 or
128 channels go 16 tokens at a time on the matrix cores (`in_chunks`), other long prompts that would leave the chip idle are
cut into pieces that are walked side by side (`pieces_for`).  The reference has no recurrent mixer of this form.
"""
from __future__ import annotations

import os
from typing import Dict, List, Optional, Tuple

import torch

from .. import kernels as K
from ..cache import StateNeed
from ..errors import ConfigError, StepError
from ..weights import TensorSpec
from .base import Mixer, MixerContext, Runtime, register_part
from .linear import fused_layout, linear, stream_layout


def pieces_for(step, units_per_sequence: int, min_piece: int) -> int:
    """Into how many pieces a step's sequences are cut so that a recurrence's walk fills the chip: a workgroup walks 16
    columns of a head's state for one sequence (`units_per_sequence` of them a sequence), and a lone prompt of a small
    model has a few dozen.  One piece (the plain walk) for single tokens, short steps and batches that fill the chip."""
    if step.is_decode or step.max_new < 4 * min_piece:
        return 1
    # a workgroup is four waves, one to a SIMD, and a lone wave waits out every latency of its token loop, so
    # pieces are asked for until four workgroups share a compute unit (BRAIDINFER_GLR_FILL, for measurements;
    # a prompt of 8,192 tokens through 8 HGRN2 layers of width 2,048 / 4,096: 17.8 / 43.3 ms at 1, 13.7 / 40.2 at 2,
    # 12.9 / 38.4 at 4, 12.8 / 38.1 at 8)
    units = step.n_seqs * units_per_sequence
    want = (int(os.environ.get("BRAIDINFER_GLR_FILL", "4")) * K.device_cus()) // max(1, units)
    return max(1, min(want, step.max_new // min_piece, 16, 65535 // max(1, step.n_seqs)))


# From this many tokens of a sequence a prompt is walked 16 tokens at a time on the matrix cores.  us against the walk token by token, in
# pieces where it can be: HGRN2, 32 heads of 128 x 128: 48 tokens 16 / 13, 64 tokens 17 / 16, 96 tokens 19 / 23, 128 tokens 21 / 28, 512
# tokens 44 / 102, 2,048 tokens 123 / 307, 3,517 and 1,501 tokens 302 / 948; WKV, 64 heads of 64 x 64: 64 tokens 16 / 17, 96 tokens 18 / 23,
# 512 tokens 38 / 76, 2,048 tokens 106 / 235; a fixed decay a head: 64 tokens 17 / 15, 96 tokens 19 / 21, 2,048 tokens 125 / 299, 1,307, 804
# and 301 tokens 162 / 295; delta rule: 64 tokens 26 / 20, 96 tokens 29 / 28, 128 tokens 32 / 36, 2,048 tokens 190 / 517, 1,307, 804 and 301
# tokens 260 / 382.  One line for all, where the delta rule's lies.  A short prompt beside longer ones would be nearly free in their chunks
# and is walked behind them (200, 153, 107 and 60 tokens: HGRN2 73 us, 50 all in chunks), the price of bits that do not depend on what is
# beside it; the line is not lowered for that, as gated outputs of 48 tokens round up to 1.16 times as far off in chunks as in the walk.
CHUNKS_FROM = 96


# A recurrence that can be walked in pieces goes so, and not in chunks, where its prompt can be cut into this many: a lone prompt
# through few heads leaves most compute units idle behind a chain of chunks, which the pieces fill.  Chunks against pieces, us: 1 to 4 heads
# of 128 x 128, 16 pieces: 2,048 tokens 100 / 80 to 110, 8,192 tokens 358 / 200 to 240, 30,000 tokens 1,254 / 570 to 670; 8 heads, 16
# pieces: 106 / 130, 368 / 340, 1,333 / 1,090; 16 heads, 8 pieces: 108 / 180, 404 / 595, 1,442 / 2,100; heads of 64 x 64: 16 of them, 16
# pieces: 86 / 75 to 88, 296 / 200 to 260; 32, 8 pieces: 89 / 110 to 136, 331 / 346 to 490; 600 tokens, 4 pieces: 39 to 44 / 50 to 82.
PIECES_FROM = 12


def in_chunks(step, d: int, e: int, pieces: int = 1) -> Tuple[bool, bool, dict]:
    """(whether sequences of the step go in chunks, whether others are walked token by token, how the walk is told apart):
    every sequence by its own number of tokens, so that what is beside it in the step does not change its bits (but for steps in
    pieces, of which the whole step decides), and the single tokens of running requests do not pay for whole chunks (a prompt of 96
    tokens among 63 of them, 32 heads of 128 x 128: delta rule 87 us so, 227 all in chunks, 323 all token by token; 16 prompts of 60
    tokens beside one of 1,500: 269, 358 and 608, a fixed decay 223, 212 and 502)."""
    if step.is_decode or step.max_new < CHUNKS_FROM or not K.chunk_takes(d, e) or pieces >= PIECES_FROM:
        return False, True, {}
    rest = [n for n in step.host_new if n < CHUNKS_FROM]
    return True, bool(rest), {"below": CHUNKS_FROM, "singles": max(rest, default=0) <= 1}


# Bytes of scratch for the chunks' factors, which are 36 KB a token for 32 heads of 128 x 128 (delta rule 68 KB) and stay with the
# engine: longer steps are taken in runs of chunks, each of which reads and writes the states once (one of 16,384 tokens:
# HGRN2 921 us, all at once 907; delta rule 1,420 and 1,380).
CHUNK_SCRATCH = 512 << 20


def chunk_scratch(step, H: int, d: int, e: int, delta: bool = False) -> dict:
    """`scratch`, and the arguments of `chunk_scan` that say which sequences it is for."""
    longs = sum(n >= CHUNKS_FROM for n in step.host_new)
    floats = min(K.chunk_scratch_floats(step.n_tokens, step.n_seqs, H, d, e, delta),
                 max(CHUNK_SCRATCH // 4, longs * K.chunk_block_floats(H, d, e, delta)))
    return {"scratch": step.ws.get("chunk_scratch", (floats,), torch.float32), "least": CHUNKS_FROM, "longs": longs}


class HGRN2(Mixer):
    graph_safe = True
    through_linear_only = True

    NAMES = {"q": "q_proj.weight", "f": "f_proj.weight", "f_bias": "f_proj.bias", "v": "v_proj.weight",
             "lower": "lower_bound", "norm": "g_norm.weight", "o": "o_proj.weight"}

    def __init__(self, hidden_size: int, num_heads: int, key_dim: int, value_dim: int, norm_eps: float,
                 names: Optional[Dict[str, str]] = None):
        if num_heads <= 0 or not 0 < key_dim <= 512 or value_dim <= 0:
            raise ConfigError(f"hgrn2: {num_heads} heads of {key_dim} query and {value_dim} value channels "
                              "(heads and widths must be positive, at most 512 query channels a head)")
        self.H, self.nh, self.d, self.e = int(hidden_size), int(num_heads), int(key_dim), int(value_dim)
        self.eps = float(norm_eps)
        self.names = dict(self.NAMES, **(names or {}))
        self.w_qfv = self.w_o = self.f_bias = self.lower = self.norm_w = None

    def weight_specs(self, prefix: str) -> List[TensorSpec]:
        n, hd = self.names, self.nh * self.d
        return [TensorSpec(prefix + n["q"], (hd, self.H)),
                TensorSpec(prefix + n["f"], (hd, self.H)),
                TensorSpec(prefix + n["f_bias"], (hd,), kind="vector", init="normal"),
                TensorSpec(prefix + n["lower"], (hd,), kind="vector", init="normal"),
                TensorSpec(prefix + n["v"], (self.nh * self.e, self.H)),
                TensorSpec(prefix + n["norm"], (self.e,), kind="vector", init="ones"),
                TensorSpec(prefix + n["o"], (self.H, self.nh * self.e))]

    def load(self, tensors: Dict[str, torch.Tensor], prefix: str, rt: Runtime) -> None:
        self.rt = rt
        n = self.names
        self.w_qfv = fused_layout([tensors[prefix + n[x]] for x in ("q", "f", "v")], rt)
        self.w_o = stream_layout(tensors[prefix + n["o"]], rt)
        self.f_bias = rt.own(tensors[prefix + n["f_bias"]].to(torch.float32))
        self.lower = rt.own(tensors[prefix + n["lower"]].to(torch.float32))
        self.norm_w = rt.own(tensors[prefix + n["norm"]].to(torch.float32))

    def state_need(self) -> StateNeed:
        return StateNeed(K.glr_state_shape(self.nh, self.d, self.e), torch.float32)

    MIN_PIECE = 128          # tokens: shorter pieces do not pay for the second walk

    def pieces_for(self, step) -> int:
        return pieces_for(step, self.nh * -(-self.e // 16), self.MIN_PIECE)

    @staticmethod
    def _piece_arrays(step, pieces: int):
        """(cuts of the packed tokens [B * pieces + 1], piece numbers [B * pieces]) on the device, made once per step
        and number of pieces: sequence b's tokens in `pieces` runs of equal length (a multiple of 16), the last ones
        shorter or empty."""
        key = ("glr_pieces", pieces)
        if key not in step.extras:
            cu, numbers, at = [0], [], 0
            for b, n in enumerate(step.host_new):
                run = -(-(-(-n // pieces)) // 16) * 16
                for c in range(pieces):
                    cu.append(at + min(n, (c + 1) * run))
                    numbers.append(b * pieces + c if step.host_slots[b] >= 0 else -1)
                at += n
            dev = torch.tensor(cu + numbers, dtype=torch.int32).to(step.tokens.device)
            step.extras[key] = (dev[:len(cu)], dev[len(cu):])
        return step.extras[key]

    def forward(self, h, x, step, ctx: MixerContext) -> None:
        T, nh, d, e = step.n_tokens, self.nh, self.d, self.e
        if ctx.state is None:
            raise StepError("hgrn2: the cache gave this mixer no state")
        # float sums of the three projections: the gates and the recurrence work on them unrounded
        rows = step.ws.get("glr_qfv", (T, 2 * nh * d + nh * e), torch.float32)
        linear(h, self.w_qfv, rows, step.ws)
        o = step.ws.get("glr_o", (T, nh * e), torch.float32)
        on = step.ws.get("glr_on", (T, nh * e), self.rt.dtype)
        one_launch = step.is_decode and T == step.n_seqs and K.head_token_takes(d, e, rows, self.f_bias, self.lower, self.norm_w, on)
        pieces = self.pieces_for(step)
        chunks, walk, rest = in_chunks(step, d, e, pieces)
        if chunks:
            hd = nh * d
            K.chunk_scan("glr", rows[:, :hd], rows[:, hd:2 * hd], rows[:, 2 * hd:], o, ctx.state, step.cu_seqlens, step.slots,
                         B=step.n_seqs, H=nh, G=nh, d=d, e=e, max_new=step.max_new, b1=self.f_bias, b2=self.lower,
                         **chunk_scratch(step, nh, d, e))
        elif pieces > 1:
            cu, numbers = self._piece_arrays(step, pieces)
            n = step.n_seqs * pieces
            piece_state = step.ws.get("glr_piece_state", (n,) + tuple(K.glr_state_shape(nh, d, e)), torch.float32)
            decay = step.ws.get("glr_decay", (n, nh, 16 * K.glr_rows_per_lane(d)), torch.float32)
            K.glr_scan_pieces(rows, self.f_bias, self.lower, o, ctx.state, step.slots, cu, numbers, piece_state, decay,
                              step.n_seqs, pieces, nh, d, e)
        if walk and (chunks or pieces == 1):
            K.glr_scan(rows, self.f_bias, self.lower, o, ctx.state, step.cu_seqlens, step.slots, step.n_seqs, nh, d, e,
                       normed=(self.norm_w, on, self.eps) if one_launch else None, **rest)
        if not one_launch:
            K.head_rmsnorm(o, self.norm_w, on, nh, e, self.eps)
        linear(on, self.w_o, x, step.ws, accumulate=True)


register_part("mixer", "hgrn2", HGRN2, replace=True)
