"""The recurrences over prompts in chunks of 16 tokens, against a float64 walk token by token and the kernels that walk so."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def walk(form, i, S, cu, H, G, d, e):
    """float64: o [T, H, e] and the last states [B, H, d, e]."""
    i = {n: x.double().cpu() if torch.is_tensor(x) else x for n, x in i.items()}
    T = i["q"].shape[0]
    q, k = (i[n].reshape(T, G, d).repeat_interleave(H // G, 1) for n in "qk")
    v = i["v"].reshape(T, H, e)
    silu = lambda x: x * torch.sigmoid(x)
    beta = None
    if form == "glr":
        low = i["b2"].reshape(H, d)
        w = low + (1 - low) * torch.sigmoid(k + i["b1"].reshape(H, d))
        q, k = silu(q), 1 - w
    elif form == "wkv":
        w = torch.exp(-torch.exp(i["z"].reshape(T, H, d) + i["b1"].reshape(H, d)))
    elif form == "fixed":
        w = i["b1"].reshape(1, H, 1).expand(T, H, d)
        if i.get("silu"):
            q, k, v = silu(q), silu(k), silu(v)
    else:
        w = i["gc"].reshape(T, H, d) if "gc" in i else i["gb"][:, :H, None].expand(T, H, d)
        beta = i["gb"][:, H:]
    o = torch.zeros(T, H, e, dtype=torch.float64)
    S = S.double().cpu().clone()
    for s in range(len(cu) - 1):
        for t in range(cu[s], cu[s + 1]):
            new = w[t][:, :, None] * S[s]
            u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.einsum("hde,hd->he", new, k[t]))
            kv = k[t][:, :, None] * u[:, None, :]
            o[t] = torch.einsum("hd,hde->he", q[t], S[s] + i["b2"].reshape(H, d)[:, :, None] * kv if form == "wkv" else new + kv)
            S[s] = new + kv
    return o, S


def inputs(form, T, H, G, d, e, strong, g):
    """Float rows as views of wider ones, and the form's vectors."""
    r = lambda *s: torch.randn(*s, generator=g) * (4.0 if strong else 1.0)
    if form in ("glr", "wkv"):
        rows = r(T, 3 * H * d + H * e + 4)
        i = {"q": rows[:, :H * d], "k": rows[:, H * d:2 * H * d], "v": rows[:, 2 * H * d:2 * H * d + H * e]}
        i["b1"] = torch.randn(H * d, generator=g) * (2.0 if strong else 0.3)
        i["b2"] = torch.rand(H * d, generator=g) * 0.5 if form == "glr" else torch.randn(H * d, generator=g)
        if form == "wkv":
            i["z"] = rows[:, 2 * H * d + H * e:3 * H * d + H * e]
        return i
    if form == "fixed":
        rows = r(T, 2 * H * d + H * e)
        return {"q": rows[:, :H * d], "k": rows[:, H * d:2 * H * d], "v": rows[:, 2 * H * d:], "silu": strong,
                "b1": torch.rand(H, generator=g) if strong else 1 - torch.rand(H, generator=g) * 0.1}
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    q, k = (unit(torch.randn(T, G, d, generator=g) + (1.0 if strong else 0.0)).reshape(T, G * d) for _ in range(2))
    gb = torch.rand(T, 2 * H, generator=g) ** (0.2 if strong else 1.0)
    i = {"q": q, "k": k, "v": r(T, H * e), "gb": gb}
    if form == "channels":
        i["gc"] = torch.rand(T, H * d, generator=g) ** (0.1 if strong else 1.0)
    return i


def as_kept(S, d):
    """[B, H, d, e] in the layout of a slot: [head][column block of 4][row % RPL][16 (column % 4) + row / RPL]."""
    B, H, _, e = S.shape
    rpl = d // 16
    return S.reshape(B, H, 16, rpl, e // 4, 4).permute(0, 1, 4, 3, 5, 2).reshape(B, H, e // 4, rpl, 64).contiguous()


# one token, a chunk less one, exactly, and one more, the ring's stages and beyond; widths of both kinds; a sequence whose slot is
# negative; decays from nearly nothing to nearly one
@pytest.mark.parametrize("form", ["glr", "wkv", "fixed", "delta", "channels"])
@pytest.mark.parametrize("d,e,H,lens,strong", [(64, 64, 3, (1, 15, 16, 17), False), (128, 128, 2, (31, 32, 48, 3), False),
                                               (64, 16, 2, (49, 64, 65, 80, 97), True), (128, 48, 1, (200,), True), (128, 16, 8, (5, 333), False),
                                               (128, 128, 40, (33, 18), True), (64, 64, 130, (35,), False)])
def test_chunks_against_token_by_token(form, d, e, H, lens, strong):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + d)
    B, T, G = len(lens), sum(lens), H // 2 if form == "delta" and H % 2 == 0 else H
    cu = np.concatenate([[0], np.cumsum(lens)]).tolist()
    he = H * e
    i = inputs(form, T, H, G, d, e, strong, g)
    form = "delta" if form == "channels" else form
    S = torch.randn(B, H, d, e, generator=g)
    want_o, want_S = walk(form, i, S, cu, H, G, d, e)
    shape = K.glr_state_shape(H, d, e)
    state = torch.full((B + 2,) + tuple(shape), 7.0, device="cuda")
    slots = torch.arange(B, dtype=torch.int32) + 1
    state[1:B + 1] = as_kept(S, d).reshape((B,) + tuple(shape)).cuda()
    out = torch.full((T, he), 7.0, device="cuda")
    scratch = torch.full((K.chunk_scratch_floats(T, B, H, d, e, form == "delta"),), float("nan"), device="cuda")
    dcu = torch.tensor(cu, dtype=torch.int32).cuda()

    def on_device():                    # with the strides of the views
        base = {}
        def put(x):
            b = x._base if x._base is not None else x
            if id(b) not in base:
                base[id(b)] = b.cuda()
            return base[id(b)].as_strided(x.shape, x.stride(), x.storage_offset())
        return {n: put(x) if torch.is_tensor(x) else x for n, x in i.items()}

    def chunks(where, st, sl):
        a = on_device()
        K.chunk_scan(form, a.pop("q"), a.pop("k"), a.pop("v"), where, st, dcu, sl.cuda(), scratch, B, H, G, d, e, max(lens), **a)
    chunks(out, state, slots)
    # float sums of at most T + d terms; the gates' own instructions are good to about an ulp of their argument's exponential
    got = out.double().cpu().reshape(T, H, e)
    assert float((got - want_o).abs().max()) < 3e-5 * float(want_o.abs().max())
    kept = as_kept(want_S.float(), d).reshape((B,) + tuple(shape))
    assert float((state[1:B + 1].cpu() - kept).abs().max()) < 3e-5 * float(kept.abs().max())
    assert torch.all(state[0] == 7.0) and torch.all(state[B + 1] == 7.0)
    # no further off than the walk token by token
    state2, out2 = torch.zeros_like(state), torch.zeros_like(out)
    state2[1:B + 1] = as_kept(S, d).reshape((B,) + tuple(shape)).cuda()
    a = on_device()
    if form == "glr":
        K.glr_scan(torch.cat([a["q"], a["k"], a["v"]], 1), a["b1"], a["b2"], out2, state2, dcu, slots.cuda(), B, H, d, e)
    elif form == "wkv":
        K.wkv_scan(torch.cat([a["q"], a["k"], a["v"], a["z"]], 1), a["b1"], a["b2"], out2, state2.reshape(B + 2, -1), dcu, slots.cuda(), B, H, d, e)
    elif form == "fixed":
        K.dr_scan(a["q"], a["k"], a["v"], None, a["b1"], out2, state2, dcu, slots.cuda(), B, H, G, d, e, silu=a["silu"])
    else:
        K.dr_scan(a["q"], a["k"], a["v"], a["gb"], None, out2, state2, dcu, slots.cuda(), B, H, G, d, e, gc=a.get("gc"))
    err = lambda x: float((x.double().cpu().reshape(T, H, e) - want_o).norm())
    assert err(out) < 1.5 * err(out2) + 1e-7 * float(want_o.norm())
    # a padding sequence: its state is left alone, its rows are zeros where the walk token by token writes zeros
    slots[0] = -1
    out.fill_(7.0)
    before = state.clone()
    chunks(out, state, slots)
    assert torch.equal(state[1], before[1]) and torch.all(out[:lens[0]] == (7.0 if form == "glr" else 0.0))


def test_values_beyond_4_gb():
    """Values as columns of rows so wide that a prompt's reach over more than 4 GB: the same bits as of dense rows."""
    from braidinfer_amd import kernels as K
    T, H, d, e, wide = 300, 1, 64, 32, 2 ** 22
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(T, H * n, device="cuda", generator=g) for n in (d, d, e))
    rows = torch.empty(T, wide, device="cuda")
    rows[:, 8:8 + H * e] = v
    decay, cu, slots = torch.full((H,), 0.95, device="cuda"), torch.tensor([0, T], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    got = []
    for x in (v, rows[:, 8:8 + H * e]):
        out, state = torch.zeros(T, H * e, device="cuda"), torch.zeros((1,) + tuple(K.glr_state_shape(H, d, e)), device="cuda")
        scratch = torch.empty(K.chunk_scratch_floats(T, 1, H, d, e), device="cuda")
        K.chunk_scan("fixed", q, k, x, out, state, cu, slots, scratch, 1, H, H, d, e, T, b1=decay)
        got.append((out, state))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and got[0][0].abs().max() > 0


@pytest.mark.parametrize("form", ["glr", "wkv", "fixed", "delta"])
@pytest.mark.parametrize("d,e", [(64, 16), (64, 64), (128, 128)])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_values_that_are_not_finite_show_from_their_token_on(form, d, e, bad):
    """An infinite value, one that is not a number, at a token of a chunk: the tokens before it and the other columns keep their
    bits, its own column shows it from its token on, as the walk token by token has it.  The same for a key, whose head shows it."""
    from braidinfer_amd import kernels as K
    T, H = 40, 2
    g = torch.Generator().manual_seed(d + e)
    i = {n: x.clone().cuda() if torch.is_tensor(x) else x for n, x in inputs(form, T, H, H, d, e, False, g).items()}
    cu, slots = torch.tensor([0, T], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()

    def run(**other):
        a = dict(i, **other)
        q, k, v = a.pop("q"), a.pop("k"), a.pop("v")
        out, state = torch.zeros(T, H * e, device="cuda"), torch.zeros((1,) + tuple(K.glr_state_shape(H, d, e)), device="cuda")
        scratch = torch.empty(K.chunk_scratch_floats(T, 1, H, d, e, form == "delta"), device="cuda")
        if form == "wkv":                                    # q, k and z share a row stride
            wide = torch.cat([q, k, a["z"]], 1)
            q, k, a["z"] = (wide[:, n * H * d:(n + 1) * H * d] for n in range(3))
        K.chunk_scan(form, q, k, v, out, state, cu, slots, scratch, 1, H, H, d, e, T, **a)
        return out
    clean = run()
    assert clean.isfinite().all()
    for t in (0, 5, 15, 16, 22, 35, 39):
        c = (7 * t + 3) % e + e * (t % 2)
        v = i["v"].clone()
        v[t, c] = bad
        got = run(v=v)
        assert not got[t:, c].isfinite().any() and torch.equal(got[:t, c], clean[:t, c])
        rest = torch.arange(H * e, device="cuda") != c
        assert torch.equal(got[:, rest], clean[:, rest])
        if form == "glr" and bad == float("inf"):            # a gate's sum of plus infinity is a decay of one
            continue
        k = i["k"].clone()
        k[t, d * (t % 2) + 9] = bad
        got = run(k=k)
        head = slice(e * (t % 2), e * (t % 2) + e)
        assert torch.equal(got[:t], clean[:t])
        if bad != bad:
            assert not got[t + 1:, head].isfinite().any()


@pytest.mark.parametrize("form", ["glr", "wkv", "fixed", "delta", "channels"])
@pytest.mark.parametrize("decay", ["slow", "middle", "fast"])
@pytest.mark.parametrize("T", [96, 1001])
def test_error_beside_the_walk_token_by_token(form, decay, T):
    """Rounding errors of chunks and of the walk token by token against float64, for decays near one, between and near zero."""
    from braidinfer_amd import kernels as K
    H, d = 4, 64 if form == "wkv" else 128
    e, x = d, {"slow": 1, "middle": 0, "fast": -1}[decay]
    g = torch.Generator(device="cuda").manual_seed(T + x)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    u = lambda *s: torch.rand(*s, device="cuda", generator=g)
    q, k, v, a = r(T, H * d), r(T, H * d), r(T, H * e), {}
    if form == "glr":
        a = {"b1": r(H * d) * 0.3 + 3 * x, "b2": u(H * d) * 0.3}
    elif form == "wkv":
        a = {"z": r(T, H * d), "b1": r(H * d) * 0.3 - 3 * x, "b2": r(H * d)}
    elif form == "fixed":
        a = {"b1": 1 - u(H) * {1: 0.01, 0: 0.2, -1: 0.9}[x]}
    else:
        q, k = (torch.nn.functional.normalize(y.view(T, H, d), dim=-1).reshape(T, H * d) for y in (q, k))
        power = {1: 0.02, 0: 0.3, -1: 2.0}[x]
        a = {"gb": torch.cat([u(T, H) ** power, u(T, H)], 1)}
        if form == "channels":
            a["gc"] = u(T, H * d) ** power
    form = "delta" if form == "channels" else form
    # float64, on the device
    D = {n: y.double() for n, y in a.items()}
    q64, k64, v64, beta = q.double().view(T, H, d), k.double().view(T, H, d), v.double().view(T, H, e), None
    if form == "glr":
        low = D["b2"].view(H, d)
        w = low + (1 - low) * torch.sigmoid(k64 + D["b1"].view(H, d))
        q64, k64 = q64 * torch.sigmoid(q64), 1 - w
    elif form == "wkv":
        w = torch.exp(-torch.exp(D["z"].view(T, H, d) + D["b1"].view(H, d)))
    elif form == "fixed":
        w = D["b1"].view(1, H, 1).expand(T, H, d)
    else:
        w, beta = D["gc"].view(T, H, d) if "gc" in D else D["gb"][:, :H, None].expand(T, H, d), D["gb"][:, H:]
    S, want = torch.zeros(H, d, e, dtype=torch.float64, device="cuda"), torch.empty(T, H, e, dtype=torch.float64, device="cuda")
    for t in range(T):
        old, S = S, w[t][:, :, None] * S
        write = v64[t] if beta is None else beta[t][:, None] * (v64[t] - (S * k64[t][:, :, None]).sum(1))
        kv = k64[t][:, :, None] * write[:, None, :]
        S = S + kv
        want[t] = (q64[t][:, :, None] * (old + D["b2"].view(H, d)[:, :, None] * kv if form == "wkv" else S)).sum(1)
    want_S = as_kept(S[None], d)[0]
    cu, slots = torch.tensor([0, T], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()

    def error(chunks):
        out, state = torch.empty(T, H * e, device="cuda"), torch.zeros((1,) + tuple(K.glr_state_shape(H, d, e)), device="cuda")
        if chunks:
            scratch = torch.empty(K.chunk_scratch_floats(T, 1, H, d, e, form == "delta"), device="cuda")
            K.chunk_scan(form, q, k, v.clone(), out, state, cu, slots, scratch, 1, H, H, d, e, T, **a)
        elif form == "glr":
            K.glr_scan(torch.cat([q, k, v], 1), a["b1"], a["b2"], out, state, cu, slots, 1, H, d, e)
        elif form == "wkv":
            K.wkv_scan(torch.cat([q, k, v, a["z"]], 1), a["b1"], a["b2"], out, state.view(1, -1), cu, slots, 1, H, d, e)
        else:
            K.dr_scan(q, k, v, a.get("gb"), a.get("b1"), out, state, cu, slots, 1, H, H, d, e, gc=a.get("gc"))
        return (float((out.double().view(T, H, e) - want).norm() / want.norm()),
                float((state.double().view(want_S.shape) - want_S).norm() / want_S.norm()))
    (out, state), (out_walk, state_walk) = error(True), error(False)
    # no further off but for what the draw does to sums of roundings (0.425 2^-24 of the norm each); a state of which little is older
    # than its last token is at most five of them: the value or its correction, the write factor, their product and two sums
    assert out < 1.12 * out_walk, (out, out_walk)
    assert state < max(1.12 * state_walk, 2 ** -24), (state, state_walk)


@pytest.mark.parametrize("form", ["glr", "wkv", "fixed", "delta", "channels"])
@pytest.mark.parametrize("lens", [(96, 1, 1, 200, 1), (95, 130, 96, 2, 1), (1, 1, 97)])
def test_long_sequences_in_chunks_beside_others_token_by_token(form, lens):
    """The two launches of a mixed step, each over its own sequences: the bits of each kernel over all of them."""
    from braidinfer_amd import kernels as K
    H, d, e, T, B = 3, 64, 32, sum(lens), len(lens)
    g = torch.Generator().manual_seed(T)
    i = {n: x.cuda() if torch.is_tensor(x) else x for n, x in inputs(form, T, H, H, d, e, False, g).items()}
    form = "delta" if form == "channels" else form
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32).cuda()
    slots = torch.arange(B, dtype=torch.int32).cuda()
    slots[-2] = -1                                           # a padding sequence
    first = torch.randn((B,) + tuple(K.glr_state_shape(H, d, e)), generator=g).cuda()
    scratch = torch.empty(K.chunk_scratch_floats(T, B, H, d, e, form == "delta"), device="cuda")
    wide = torch.cat([i["q"], i["k"], i["v"]] + ([i["z"]] if form == "wkv" else []), 1).contiguous()
    hd, he = H * d, H * e
    q, k, v = wide[:, :hd], wide[:, hd:2 * hd], wide[:, 2 * hd:2 * hd + he]
    rest = {n: x for n, x in i.items() if n not in ("q", "k", "v", "z")}

    def chunks(out, state, least):
        z = {"z": wide[:, 2 * hd + he:]} if form == "wkv" else {}
        K.chunk_scan(form, q, k, v, out, state, cu, slots, scratch, B, H, H, d, e, max(lens), least=least, **z, **rest)

    def walk(out, state, **kw):
        if form == "glr":
            K.glr_scan(wide, i["b1"], i["b2"], out, state, cu, slots, B, H, d, e, **kw)
        elif form == "wkv":
            kw.pop("singles", None)
            K.wkv_scan(wide, i["b1"], i["b2"], out, state.view(B, -1), cu, slots, B, H, d, e, **kw)
        else:
            K.dr_scan(q, k, v, i.get("gb"), i.get("b1"), out, state, cu, slots, B, H, H, d, e, gc=i.get("gc"), **kw)

    def run(*calls):
        out, state = torch.full((T, he), 7.0, device="cuda"), first.clone()
        for call in calls:
            call(out, state)
        return out, state
    whole, token = run(lambda o, s: chunks(o, s, 0)), run(lambda o, s: walk(o, s))
    few = max(n for n in lens if n < 96) <= 1
    both = run(lambda o, s: chunks(o, s, 96), lambda o, s: walk(o, s, below=96, singles=few))
    for b, n in enumerate(lens):
        want, at = (whole if n >= 96 else token), slice(int(cu[b]), int(cu[b + 1]))
        assert torch.equal(both[0][at], want[0][at]) and torch.equal(both[1][b], want[1][b]), (b, n)


@pytest.mark.parametrize("form", ["glr", "wkv", "fixed", "delta"])
def test_chunks_in_runs_where_the_scratch_is_small(form):
    """Fewer chunks at once: the same bits, nothing written behind the scratch, too little of it refused."""
    from braidinfer_amd import kernels as K
    from braidinfer_amd.errors import KernelError
    H, d, e, lens = 3, 64, 32, (400, 1, 130, 96, 20, 97)
    T, B, longs = sum(lens), len(lens), 4
    g = torch.Generator().manual_seed(5)
    i = {n: x.cuda() if torch.is_tensor(x) else x for n, x in inputs(form, T, H, H, d, e, form == "fixed", g).items()}
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32).cuda()
    slots = torch.arange(B, dtype=torch.int32).cuda()
    slots[2] = -1
    first = torch.randn((B,) + tuple(K.glr_state_shape(H, d, e)), generator=g).cuda()
    wide = torch.cat([i["q"], i["k"], i["v"]] + ([i["z"]] if form == "wkv" else []), 1).contiguous()
    hd, he, block = H * d, H * e, K.chunk_block_floats(H, d, e, form == "delta")
    rest = {n: x for n, x in i.items() if n not in ("q", "k", "v", "z")}

    def run(floats, **kw):
        rows = wide.clone()                                  # silu goes back into the values
        if form == "wkv":
            kw["z"] = rows[:, 2 * hd + he:]
        out, state, scratch = torch.full((T, he), 7.0, device="cuda"), first.clone(), torch.full((floats + 64,), 5.0, device="cuda")
        K.chunk_scan(form, rows[:, :hd], rows[:, hd:2 * hd], rows[:, 2 * hd:2 * hd + he], out, state, cu, slots, scratch[:floats], B, H, H, d, e,
                     max(lens), least=96, **kw, **rest)
        assert torch.all(scratch[floats:] == 5.0)
        return out, state
    want = run(K.chunk_scratch_floats(T, B, H, d, e, form == "delta"))
    assert torch.all(want[0][400] == 7.0) and torch.equal(want[1][1], first[1]) and not torch.equal(want[1][5], first[5])
    for chunks in (1, 2, 5, 6, 7, 24):
        for got in (run(longs * chunks * block + 40, longs=longs), run(B * chunks * block)):
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with pytest.raises(KernelError):
        run(longs * block - 4, longs=longs)


# heads in steps of 8 and not; the longest sequence first, last and between, equal ones, more sequences than are ordered; a padding sequence among them
@pytest.mark.parametrize("form,d,H", [("glr", 64, 8), ("fixed", 128, 8), ("delta", 128, 8), ("wkv", 64, 16), ("delta", 64, 12)])
@pytest.mark.parametrize("lens", [[200, 40, 97, 16], [16, 40, 97, 200], [33, 180, 33, 180, 1], [17 + i % 3 for i in range(66)], [300, 20, 20, 20, 20, 20, 20]])
def test_a_sequences_bits_do_not_depend_on_the_others(form, d, H, lens):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(len(lens) + d)
    T, B, e = sum(lens), len(lens), 32
    i = {n: x.cuda() if torch.is_tensor(x) else x for n, x in inputs(form, T, H, H, d, e, False, g).items()}
    n = 1
    for x in K.glr_state_shape(H, d, e):
        n *= x
    first = torch.randn(B, n, generator=g).cuda()
    cu = np.concatenate([[0], np.cumsum(lens)]).tolist()
    vectors = {name: i[name] for name in ("b1", "b2") if name in i}
    slots = [b if b != 1 else -1 for b in range(B)]

    def run(t0, t1, some, state):
        rows = {name: i[name][t0:t1] for name in ("z", "gb", "gc") if name in i}
        at = [c - t0 for c in cu if t0 <= c <= t1]
        o = torch.full((t1 - t0, H * e), 7.0, device="cuda")
        scratch = torch.empty(K.chunk_scratch_floats(t1 - t0, len(some), H, d, e, form == "delta"), device="cuda")
        K.chunk_scan(form, i["q"][t0:t1], i["k"][t0:t1], i["v"][t0:t1].clone(), o, state, torch.tensor(at, dtype=torch.int32, device="cuda"),
                     torch.tensor(some, dtype=torch.int32, device="cuda"), scratch, len(some), H, H, d, e, max(b - a for a, b in zip(at, at[1:])), **rows, **vectors)
        return o
    together, alone = first.clone(), first.clone()
    o = run(0, T, slots, together)
    for b in range(B):
        if slots[b] >= 0:
            assert torch.equal(run(cu[b], cu[b + 1], [b], alone), o[cu[b]:cu[b + 1]]), b
    assert torch.equal(together, alone) and torch.equal(together[1], first[1])
