"""The recurrences over prompts in chunks of 16 tokens, against a float64 walk token by token and the kernels that walk so."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def walk(form, rows, b1, b2, S, cu, H, d, e):
    """float64: o [T, H, e] and the last states [B, H, d, e]."""
    rows = rows.double().cpu()
    T, hd = rows.shape[0], H * d
    b1, b2 = b1.double().cpu().reshape(H, d), b2.double().cpu().reshape(H, d)
    q = rows[:, :hd].reshape(T, H, d)
    k = rows[:, hd:2 * hd].reshape(T, H, d)
    v = rows[:, 2 * hd:2 * hd + H * e].reshape(T, H, e)
    if form == "glr":
        w = b2 + (1 - b2) * torch.sigmoid(k + b1)
        q, k = q * torch.sigmoid(q), 1 - w
    else:
        w = torch.exp(-torch.exp(rows[:, 2 * hd + H * e:3 * hd + H * e].reshape(T, H, d) + b1))
    o = torch.zeros(T, H, e, dtype=torch.float64)
    S = S.double().cpu().clone()
    for s in range(len(cu) - 1):
        for t in range(cu[s], cu[s + 1]):
            kv = k[t][:, :, None] * v[t][:, None, :]
            new = w[t][:, :, None] * S[s] + kv
            o[t] = torch.einsum("hd,hde->he", q[t], new if form == "glr" else S[s] + b2[:, :, None] * kv)
            S[s] = new
    return o, S


def as_kept(S, d):
    """[B, H, d, e] in the layout of a slot: [head][column block of 4][row % RPL][16 (column % 4) + row / RPL]."""
    B, H, _, e = S.shape
    rpl = d // 16
    return S.reshape(B, H, 16, rpl, e // 4, 4).permute(0, 1, 4, 3, 5, 2).reshape(B, H, e // 4, rpl, 64).contiguous()


# one token, a chunk less one, exactly, and one more, the ring's stages and beyond; widths of both kinds; a sequence whose slot is
# negative; decays from nearly nothing to nearly one
@pytest.mark.parametrize("form", ["glr", "wkv"])
@pytest.mark.parametrize("d,e,H,lens,strong", [(64, 64, 3, (1, 15, 16, 17), False), (128, 128, 2, (31, 32, 48, 3), False),
                                               (64, 16, 2, (49, 64, 65, 80, 97), True), (128, 48, 1, (200,), True), (128, 16, 8, (5, 333), False)])
def test_chunks_against_token_by_token(form, d, e, H, lens, strong):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + d)
    B, T = len(lens), sum(lens)
    cu = np.concatenate([[0], np.cumsum(lens)]).tolist()
    hd, he = H * d, H * e
    width = 2 * hd + he if form == "glr" else 3 * hd + he + 4
    rows = torch.randn(T, width, generator=g) * (4.0 if strong else 1.0)
    b1 = torch.randn(hd, generator=g) * (2.0 if strong else 0.3)
    b2 = torch.rand(hd, generator=g) * 0.5 if form == "glr" else torch.randn(hd, generator=g)
    S = torch.randn(B, H, d, e, generator=g)
    want_o, want_S = walk(form, rows, b1, b2, S, cu, H, d, e)
    shape = K.glr_state_shape(H, d, e)
    state = torch.full((B + 2,) + tuple(shape), 7.0, device="cuda")
    slots = torch.arange(B, dtype=torch.int32) + 1
    state[1:B + 1] = as_kept(S, d).reshape((B,) + tuple(shape)).cuda()
    out = torch.full((T, he), 7.0, device="cuda")
    scratch = torch.full((K.chunk_scratch_floats(T, B, H, d),), float("nan"), device="cuda")
    args = (rows.cuda(), b1.cuda(), b2.cuda())
    dcu = torch.tensor(cu, dtype=torch.int32).cuda()
    flat = state if form == "glr" else state.reshape(B + 2, -1)
    K.chunk_scan(form, *args, out, flat, dcu, slots.cuda(), scratch, B, H, d, e, max(lens))
    # float sums of at most T + d terms; the gates' own instructions are good to about an ulp of their argument's exponential
    got = out.double().cpu().reshape(T, H, e)
    assert float((got - want_o).abs().max()) < 3e-5 * float(want_o.abs().max())
    kept = as_kept(want_S.float(), d).reshape((B,) + tuple(shape))
    assert float((state[1:B + 1].cpu() - kept).abs().max()) < 3e-5 * float(kept.abs().max())
    assert torch.all(state[0] == 7.0) and torch.all(state[B + 1] == 7.0)
    # no further off than the walk token by token
    state2, out2 = torch.zeros_like(state), torch.zeros_like(out)
    state2[1:B + 1] = as_kept(S, d).reshape((B,) + tuple(shape)).cuda()
    scan = K.glr_scan if form == "glr" else K.wkv_scan
    scan(*args, out2, state2 if form == "glr" else state2.reshape(B + 2, -1), dcu, slots.cuda(), B, H, d, e)
    err = lambda x: float((x.double().cpu().reshape(T, H, e) - want_o).norm())
    assert err(out) < 1.5 * err(out2) + 1e-7 * float(want_o.norm())
    # a padding sequence: its state is left alone, its rows are zeros where the walk token by token writes zeros
    slots[0] = -1
    out.fill_(7.0)
    before = state.clone()
    K.chunk_scan(form, *args, out, flat, dcu, slots.cuda(), scratch, B, H, d, e, max(lens))
    assert torch.equal(state[1], before[1]) and torch.all(out[:lens[0]] == (7.0 if form == "glr" else 0.0))
