"""Which products a step of routed experts goes through, by its tokens and widths: the rule alone, on the host."""
import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.errors import KernelError
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
                 "experts_up_tiles", "experts_wide", "experts_gather", "experts_gemm", "experts_combine", "silu_mul", "gemm"):
        monkeypatch.setattr(K, name, lambda *a, _name=name, **k: called.append(_name))
    monkeypatch.setattr(feedforward, "linear", lambda *a, **k: None)
    part = feedforward.RoutedExperts(W, F, E, top)
    part.rt, part.n_scores = type("Runtime", (), {"dtype": dtype}), E
    part.w_gu, part.w_down = (torch.empty(shape, dtype=dtype, device="meta") for shape in ((E, 2 * F, W), (E, W, F)))
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


FEW, GATHERED = ["experts_up_grouped", "experts_down_grouped"], ["experts_gather", "experts_gemm", "silu_mul", "experts_gemm"]
WIDE = ["experts_wide", "experts_wide"]


# 22 tokens: five and a half pairs an expert, the last that the streams take; 64 and 88: 16 and 22, the last before the tiles
@pytest.mark.parametrize("W,F,E,top,last", [(4096, 1792, 32, 8, 64), (2048, 1408, 16, 4, 88)])
def test_few_pairs_and_many(monkeypatch, W, F, E, top, last):
    for tokens, decode, want in ((1, True, FEW), (16, True, FEW), (22, True, FEW), (23, True, WIDE), (last, True, WIDE), (last + 1, True, TILES), (200, True, TILES),
                                 (17, False, FEW), (22, False, FEW), (23, False, WIDE), (47, False, WIDE), (48, False, WIDE), (last, False, WIDE),
                                 (last + 1, False, TILES), (4000, False, TILES)):
        assert route(monkeypatch, tokens, decode, W, F, E, top) == want, tokens


def test_sixteen_tokens_stay_with_the_streams(monkeypatch):
    """No expert has more than 16 of them, whatever their average."""
    for decode in (True, False):
        assert route(monkeypatch, 16, decode, E=8, top=4) == FEW and route(monkeypatch, 17, decode, E=8, top=4) == WIDE
        assert route(monkeypatch, 16, decode, E=4, top=4) == FEW and route(monkeypatch, 23, decode, E=4, top=4) == TILES


def test_each_product_by_its_own_widths(monkeypatch):
    """Widths of which one is no whole number of chunks of 128: that product stays with the streams, or with the tiles."""
    assert route(monkeypatch, 23, True, 4096, 1800) == ["experts_wide", "experts_down_grouped"]
    assert route(monkeypatch, 64, False, 4096, 1856) == ["experts_wide", "experts_gemm"]
    assert route(monkeypatch, 64, False, 4160, 1792) == ["experts_up_tiles", "experts_wide"]
    assert route(monkeypatch, 64, False, 4104, 1792) == ["experts_gather", "experts_gemm", "silu_mul", "experts_wide"]


def test_rows_off_16_bytes(monkeypatch):
    """Rows or weights that start between multiples of 16 bytes are not for `experts_wide`, and the wrappers of the kernels that take
    them call these, whatever the number of pairs."""
    E, F, W, T, top = 4, 256, 256, 20, 2
    wide, called = torch.zeros(2 * E * F * W + 8, dtype=torch.bfloat16), []
    monkeypatch.setattr(K, "_dev", lambda *a: None)
    monkeypatch.setattr(K, "_stream", lambda: 0)
    takes = K._fn("experts_wide", "br_experts_wide_takes", [K.c_int] * 4)
    monkeypatch.setattr(K, "_fn", lambda module, name, types: takes if name == "br_experts_wide_takes" else lambda *a: called.append(name) or 0)
    first, order = torch.zeros(E + 1, dtype=torch.int32), torch.zeros(T * top, dtype=torch.int32)
    y, out = torch.zeros(T * top, F, dtype=torch.bfloat16), torch.zeros(T * top, W)
    for off in (0, 4, 8):
        gu, dn = wide[off:off + 2 * E * F * W].view(E, 2 * F, W), wide[off:off + E * F * W].view(E, W, F)
        h = wide[off:off + T * W].view(T, W)
        for a, w in ((h, gu), (h.clone(), gu), (h, gu.clone()), (y, dn)):
            assert K.experts_wide_pays(a, w, T, T * top) == (a.data_ptr() % 16 == w.data_ptr() % 16 == 0)
        K.experts_up_grouped(h, gu, first, order, y, top)
        K.experts_down_grouped(y, dn, first, out, T)
    assert called == 3 * ["br_experts_up_grouped", "br_experts_down_grouped"]


def test_widths_that_the_tiles_do_not_take(monkeypatch):
    for tokens, decode, want in ((1, True, FEW), (100, True, FEW), (47, False, FEW), (48, False, GATHERED), (6143, False, GATHERED),
                                 (6144, False, GATHERED[:1])):
        assert route(monkeypatch, tokens, decode, 96, 40, 8, 2) == want, tokens
    assert route(monkeypatch, 5, False, 50, 9, 3, 2) == ["experts_up", "experts_down"]
    assert route(monkeypatch, 5, True, dtype=torch.float32) == ["experts_up", "experts_down"]
    assert route(monkeypatch, 50, False, dtype=torch.float32) == ["experts_gather"]


def test_the_forced_routes(monkeypatch):
    monkeypatch.setenv("BRAIDINFER_EXPERTS_ONE_BY_ONE", "1")
    for W, F in ((4096, 1792), (96, 40)):
        assert route(monkeypatch, 300, False, W, F) == ["experts_gather"]
        assert route(monkeypatch, 300, True, W, F) == FEW
    monkeypatch.setenv("BRAIDINFER_EXPERTS_ONE_BY_ONE", "0")
    assert route(monkeypatch, 300, False) == TILES
    assert route(monkeypatch, 100000, False, 96, 40, 8, 2) == GATHERED          # 25,000 pairs an expert, in one launch all the same


def test_all_waves_together_refuse(monkeypatch):
    """Arrays of other types or sizes than the kernel reads are an error before anything is launched."""
    E, F, W, T, top = 3, 256, 384, 9, 2
    called = []
    monkeypatch.setattr(K, "_dev", lambda *a: None)
    monkeypatch.setattr(K, "_stream", lambda: 0)
    monkeypatch.setattr(K, "_fn", lambda module, name, types: lambda *a: called.append(name) or 0)
    n = T * top
    h, gu, dn = (torch.zeros(shape, dtype=torch.bfloat16) for shape in ((T, W), (E, 2 * F, W), (E, W, F)))
    first, order = torch.zeros(E + 1, dtype=torch.int32), torch.zeros(n, dtype=torch.int32)
    y, out = torch.zeros(n, F, dtype=torch.bfloat16), torch.zeros(n, W)
    K.experts_wide(h, gu, first, order, y, top)
    K.experts_wide(y, dn, first, None, out)
    assert called == 2 * ["br_experts_wide"]
    for args in ((h, gu, first.long(), order, y, top), (h, gu, first, order.long(), y, top), (y, dn, first.long(), None, out), (h, gu, first[:E], order, y, top),
                 (h.float(), gu, first, order, y, top), (h, gu, first, order, y.float(), top), (y, dn, first, None, out.bfloat16()),
                 (h[:4], gu, first, order, y, top), (y[:4], dn, first, None, out), (h, gu, first, order[:4], y, top), (h[:, :256], gu, first, order, y, top)):
        with pytest.raises(KernelError):
            K.experts_wide(*args)
    assert len(called) == 2


def test_where_all_waves_together_end():
    """By the tiles of 256 rows that the prompt products would have: up to one to a compute unit, up to three rounds of them, beyond."""
    a = torch.empty(1, 256, dtype=torch.bfloat16, device="meta")
    for E, N, most in ((16, 4096, 22), (16, 4097, 16), (32, 4096, 16), (64, 2816, 16), (64, 3072, 10), (128, 1536, 10)):
        w = torch.empty(E, N, 256, dtype=torch.bfloat16, device="meta")
        assert K.experts_wide_pays(a, w, 17, most * E) and not K.experts_wide_pays(a, w, 17, most * E + 1), (E, N)
        assert K.experts_wide_pays(a, w, 17, 6 * E) and not K.experts_wide_pays(a, w, 16, 6 * E) and not K.experts_wide_pays(a, w, 17, 11 * E // 2)
