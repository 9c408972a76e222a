"""The routed experts' products at the edges of their kernels' tiles, against float64 products of the same bfloat16 values."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def bf(a):
    return torch.tensor(a, dtype=torch.float32).to(torch.bfloat16)


def sorted_pairs(chosen, bins):
    from braidinfer_amd import kernels as K
    n = chosen.numel()
    first, order, place = (torch.zeros(k, dtype=torch.int32, device="cuda") for k in (bins + 1, n, n))
    K.experts_sort(chosen, first, order, place, bins)
    return first, order, place


def drawn(T, top, E, how, seed):
    """[T, top] expert numbers: spread evenly, drawn, or all tokens to the last `top` experts."""
    rng = np.random.default_rng(seed)
    if how == "one":
        rows = [np.arange(E - top, E)] * T
    else:
        rows = [rng.permutation(E)[:top] for _ in range(T)]
    return torch.tensor(np.stack(rows).astype(np.int32)).cuda()


def products(h, w_gu, w_down, chosen, limit, alpha):
    """float64: (y [T, top, F], W_d y with y rounded as the kernels store it [T, top, W])."""
    h64, gu, dn = h.cuda().double(), w_gu.cuda(), w_down.cuda()
    T, top = chosen.shape
    F, W = gu.shape[1] // 2, gu.shape[2]
    y = torch.zeros(T, top, F, dtype=torch.float64, device="cuda")
    out = torch.zeros(T, top, W, dtype=torch.float64, device="cuda")
    for e in range(gu.shape[0]):
        t, s = (chosen == e).nonzero(as_tuple=True)
        if len(t):
            z = h64[t] @ gu[e].double().T
            g, u = z[:, :F], z[:, F:]
            if alpha:
                g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1.0
                v = g * torch.sigmoid(alpha * g) * u
            else:
                v = g * torch.sigmoid(g) * u
            y[t, s] = v
            out[t, s] = v.to(torch.bfloat16).double() @ dn[e].double().T
    return y, out


# widths with 8 to 33 chunks of 128 (every wave one, some two, some four); tokens at 1, around 8 and 16 pairs an expert, and
# beyond; experts without pairs, all pairs in the last experts, numbers behind the experts (identities)
@pytest.mark.parametrize("T,top,E,W,F,how,identity,alpha", [
    (1, 1, 1, 1024, 1024, "drawn", 0, 0.0), (1, 8, 32, 2048, 1408, "drawn", 0, 0.0), (6, 8, 32, 4224, 1792, "drawn", 0, 0.0),
    (8, 2, 5, 1152, 1032, "one", 0, 1.702), (9, 2, 5, 1152, 1024, "one", 0, 0.0), (16, 3, 7, 1024, 1280, "one", 0, 0.0),
    (17, 3, 70, 1024, 1152, "drawn", 3, 0.0), (40, 8, 32, 1536, 1792, "drawn", 0, 0.0), (64, 4, 16, 2048, 1408, "one", 2, 1.702),
    (64, 16, 16, 1024, 1024, "drawn", 0, 0.0)])
def test_products_of_few_tokens(T, top, E, W, F, how, identity, alpha):
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(T + W + F)
    h, w_gu, w_down = bf(rng.standard_normal((T, W))), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5), bf(rng.standard_normal((E, W, F)) / F ** 0.5)
    chosen = drawn(T, top, E + identity, how, T)
    want_y, want = products(h, w_gu, w_down, chosen, 0.9, alpha)
    first, order, place = sorted_pairs(chosen, E + (1 if identity else 0))
    hd, gu, dn = h.cuda(), w_gu.cuda(), w_down.cuda()
    n = T * top
    y = torch.full((n, F), 7.0, dtype=torch.bfloat16, device="cuda")
    K.experts_up_grouped(hd, gu, first, order, y, top, 0.9 if alpha else 0.0, alpha)
    out = torch.full((n, W), 7.0, dtype=torch.float32, device="cuda")
    K.experts_down_grouped(y, dn, first, out, T)
    real = chosen < E
    got_y, got = y[place.long()].double().reshape(T, top, F), out[place.long()].double().reshape(T, top, W)
    # y: one bfloat16 rounding (2^-9) of a value of order one; out: float sums of the same bfloat16 rows, rows that y's
    # rounding may send to a neighbour (2^-8 of single elements of a sum of F)
    assert float((got_y - want_y)[real].abs().max()) < 2 ** -8 * float(want_y.abs().max())
    assert float((got - want)[real].abs().max()) < 2 ** -7 * float(want.abs().max())
    assert float((got - want)[real].norm() / want[real].norm()) < 1e-3
    for t, s in [(0, 0), (T - 1, top - 1)]:
        if chosen[t, s] < E:                       # the product of the stored rows themselves: float sums only
            exact = dn[int(chosen[t, s])].double() @ y[place[t * top + s].long()].double()
            assert float((got[t, s] - exact).abs().max()) < 2e-6 * float(exact.abs().max()) * (F / 1024) ** 0.5 + 1e-5 * float(exact.abs().mean())


def test_rows_and_weights_off_16_bytes():
    """Rows and matrices that start 8 bytes behind a multiple of 16, at ten pairs an expert: taken, with the products of aligned ones."""
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(5)
    T, top, E, W, F = 20, 4, 8, 1024, 1152

    def shifted(t):
        room = torch.zeros(t.numel() + 4, dtype=t.dtype, device="cuda")
        room[4:] = t.reshape(-1).cuda()
        return room[4:].view(t.shape)
    h, gu, dn = bf(rng.standard_normal((T, W))), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5), bf(rng.standard_normal((E, W, F)) / F ** 0.5)
    chosen = drawn(T, top, E, "drawn", 6)
    first, order, place = sorted_pairs(chosen, E)
    want_y, want = products(h, gu, dn, chosen, 0.0, 0.0)
    for shift in ((shifted, torch.Tensor.cuda), (torch.Tensor.cuda, shifted)):
        y, out = torch.zeros((T * top, F), dtype=torch.bfloat16, device="cuda"), torch.zeros((T * top, W), device="cuda")
        K.experts_up_grouped(shift[0](h), shift[1](gu), first, order, y, top)
        K.experts_down_grouped(shift[0](y), shift[1](dn), first, out, T)
        got_y, got = y[place.long()].double().reshape(T, top, F), out[place.long()].double().reshape(T, top, W)
        assert float((got_y - want_y).abs().max()) < 2 ** -8 * float(want_y.abs().max())           # one bfloat16 rounding, 2^-9
        assert float((got - want).norm() / want.norm()) < 1e-3                                     # rows that y's rounding may send to a neighbour


def test_a_tokens_experts_do_not_depend_on_its_batch():
    """The same rows alone and among others through the streamed products: the same bits."""
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(3)
    T, top, E, W, F = 12, 4, 9, 1024, 1152
    h, gu, dn = bf(rng.standard_normal((T, W))).cuda(), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5).cuda(), bf(rng.standard_normal((E, W, F))).cuda()
    chosen = drawn(T, top, E, "drawn", 4)

    def run(k):
        first, order, place = sorted_pairs(chosen[:k].contiguous(), E)
        y = torch.zeros((k * top, F), dtype=torch.bfloat16, device="cuda")
        K.experts_up_grouped(h[:k].contiguous(), gu, first, order, y, top)
        out = torch.zeros((k * top, W), dtype=torch.float32, device="cuda")
        K.experts_down_grouped(y, dn, first, out, k)
        return out[place.long()].reshape(k, top, W)
    whole = run(T)
    for k in (1, 3, 8, 9):
        assert torch.equal(run(k), whole[:k])


# pairs an expert at 0, 1, below, at and beyond a tile's 128 and 256 rows; widths with an odd number of 64-wide steps and of 256
# output columns cut short; more than 64 experts; identities behind them
@pytest.mark.parametrize("T,top,E,W,F,how,identity,alpha", [
    (1, 1, 3, 64, 64, "drawn", 0, 0.0), (65, 2, 2, 192, 320, "one", 0, 0.0), (128, 1, 3, 64, 128, "one", 0, 1.702),
    (129, 3, 4, 320, 64, "one", 0, 0.0), (257, 2, 5, 256, 192, "one", 1, 0.0), (300, 4, 90, 128, 192, "drawn", 3, 0.0),
    (520, 2, 3, 448, 320, "drawn", 0, 0.0), (900, 8, 16, 1024, 704, "drawn", 0, 1.702)])
def test_products_of_many_tokens(T, top, E, W, F, how, identity, alpha):
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(T + W + F)
    h, w_gu, w_down = bf(rng.standard_normal((T, W))), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5), bf(rng.standard_normal((E, W, F)) / F ** 0.5)
    chosen = drawn(T, top, E + identity, how, T)
    want_y, want = products(h, w_gu, w_down, chosen, 0.9, alpha)
    first, order, place = sorted_pairs(chosen, E + (1 if identity else 0))
    n = T * top
    y = torch.full((n, F), 7.0, dtype=torch.bfloat16, device="cuda")
    K.experts_up_tiles(h.cuda(), w_gu.cuda(), first, order, y, top, 0.9 if alpha else 0.0, alpha)
    for dtype, rounding in ((torch.float32, 0.0), (torch.bfloat16, 2 ** -9)):
        out = torch.full((n, W), 7.0, dtype=dtype, device="cuda")
        K.experts_gemm(y, w_down.cuda(), first, out)
        real = chosen < E
        got_y, got = y[place.long()].double().reshape(T, top, F), out[place.long()].double().reshape(T, top, W)
        assert float((got_y - want_y)[real].abs().max()) < 2 ** -8 * float(want_y.abs().max())
        assert float((got - want)[real].abs().max()) < (2 ** -7 + rounding) * float(want.abs().max())
        assert float((got - want)[real].norm() / want[real].norm()) < 1e-3 + rounding
        if identity:                               # rows behind the experts' pairs are nobody's
            assert torch.all(out[int(first[E]):] == 7.0)


# few experts with up to a group of 64 pairs and one more; widths of 2 and 3 chunks of 128 and of no whole number of any unit's rows;
# identities behind the experts
@pytest.mark.parametrize("T,top,E,W,F,how,identity,alpha", [
    (31, 1, 1, 256, 256, "one", 0, 0.0), (32, 2, 3, 384, 256, "one", 0, 0.0), (33, 1, 2, 256, 400, "drawn", 1, 1.702), (63, 1, 2, 400, 256, "one", 0, 0.0),
    (65, 2, 4, 512, 384, "one", 0, 0.0), (40, 8, 32, 640, 1152, "drawn", 0, 0.0), (100, 3, 9, 1024, 256, "drawn", 2, 1.702), (24, 8, 32, 1024, 888, "drawn", 0, 0.0)])
def test_products_by_all_waves_together(T, top, E, W, F, how, identity, alpha):
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(T + W + F)
    h, w_gu = bf(rng.standard_normal((T, W))), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5)
    w_down = bf(rng.standard_normal((E, W, F)) / F ** 0.5)
    chosen = drawn(T, top, E + identity, how, T)
    want_y, want = products(h, w_gu, w_down, chosen, 0.9, alpha)
    first, order, place = sorted_pairs(chosen, E + (1 if identity else 0))
    n, real = T * top, chosen < E
    if W % 128 == 0:
        y = torch.full((n, F), 7.0, dtype=torch.bfloat16, device="cuda")
        K.experts_wide(h.cuda(), w_gu.cuda(), first, order, y, top, 0.9 if alpha else 0.0, alpha)
        got_y = y[place.long()].double().reshape(T, top, F)
        assert float((got_y - want_y)[real].abs().max()) < 2 ** -8 * float(want_y.abs().max())      # one bfloat16 rounding, 2^-9
        assert torch.all(y[int(first[E]):] == 7.0)                                                  # identities' rows are nobody's
    if F % 128 == 0:
        y = want_y.to(torch.bfloat16).reshape(n, F)[order.long()].contiguous()
        out = torch.full((n, W), 7.0, dtype=torch.float32, device="cuda")
        K.experts_wide(y, w_down.cuda(), first, None, out)
        got = out[place.long()].double().reshape(T, top, W)
        # float sums of the same rows: F products in any order, each of at most the largest |row| x |weight|
        assert float((got - want)[real].abs().max()) < F * 2 ** -24 * float(want_y.abs().max()) * float(w_down.abs().max())
        assert float((got - want)[real].norm() / want[real].norm()) < 1e-5
        assert torch.all(out[int(first[E]):] == 7.0)


# every height of a unit, 64 to 128 weight rows, in both products (the rule on the matrices picks it, for 256 compute units); experts of
# no pair, one, and around one and two groups of 32 and of 64; every height by groups of 32, of 64 and as the kernel chooses
@pytest.mark.parametrize("W,F,up,down", [(640, 512, 64, 64), (1664, 896, 80, 80), (2048, 1024, 96, 96), (2432, 1280, 112, 112), (2816, 1408, 128, 128)])
@pytest.mark.parametrize("few", [True, False])
def test_heights_and_groups(W, F, up, down, few):
    from braidinfer_amd import kernels as K
    counts = [31, 32, 0, 33, 1, 31, 32, 33, 7, 0] if few else [63, 64, 65, 31, 32, 33, 0, 1, 128, 129]
    E, T = len(counts), sum(counts)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (K.experts_wide_rows(E, F, True), K.experts_wide_rows(E, W, False)) == (up, down)
    g = torch.Generator(device="cuda").manual_seed(W + few)
    h, w_gu, w_down = (torch.randn(shape, generator=g, device="cuda").div(shape[-1] ** 0.5 if len(shape) > 2 else 1.0).to(torch.bfloat16)
                       for shape in ((T, W), (E, 2 * F, W), (E, W, F)))
    chosen = torch.tensor(np.random.default_rng(W + few).permutation(np.repeat(np.arange(E), counts)).astype(np.int32)).cuda().reshape(T, 1)
    want_y, want = products(h, w_gu, w_down, chosen, 0.0, 0.0)
    first, order, place = sorted_pairs(chosen, E)
    rows = want_y.to(torch.bfloat16).reshape(T, F)[order.long()].contiguous()
    got = []
    for group in (32, 64, 0):
        y, out = torch.full((T, F), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((T, W), 7.0, device="cuda")
        K.experts_wide(h, w_gu, first, order, y, 1, group=group)
        K.experts_wide(rows, w_down, first, None, out, group=group)
        got.append((y, out))
        assert torch.equal(y, got[0][0]) and torch.equal(out, got[0][1])           # a pair's sums do not depend on its group
    y, out = got[0][0][place.long()].double(), got[0][1][place.long()].double()
    assert float((y - want_y[:, 0]).abs().max()) < 2 ** -8 * float(want_y.abs().max())                           # one bfloat16 rounding, 2^-9
    # float sums of the same rows: F products in any order, each of at most the largest |row| x |weight|
    assert float((out - want[:, 0]).abs().max()) < F * 2 ** -24 * float(want_y.abs().max()) * float(w_down.abs().max())
    assert float((out - want[:, 0]).norm() / want.norm()) < 1e-6


def test_a_tokens_experts_do_not_depend_on_its_batch_among_all_waves():
    """The same rows in steps of other sizes, by groups of 32 and of 64: the same bits.  (By the streams and by these kernels a token's
    outputs differ in the order of their sums: up to 16 tokens, or five and a half pairs an expert, they are the streams'.)"""
    from braidinfer_amd import kernels as K
    rng = np.random.default_rng(8)
    T, top, E, W, F = 90, 4, 8, 512, 640
    h, gu, dn = bf(rng.standard_normal((T, W))).cuda(), bf(rng.standard_normal((E, 2 * F, W)) / W ** 0.5).cuda(), bf(rng.standard_normal((E, W, F))).cuda()
    chosen = drawn(T, top, E, "drawn", 4)

    def run(k):
        first, order, place = sorted_pairs(chosen[:k].contiguous(), E)
        y, out = torch.zeros((k * top, F), dtype=torch.bfloat16, device="cuda"), torch.zeros((k * top, W), device="cuda")
        K.experts_wide(h[:k].contiguous(), gu, first, order, y, top)
        K.experts_wide(y, dn, first, None, out)
        return out[place.long()].reshape(k, top, W)
    whole = run(T)
    for k in (1, 17, 32, 33, 64):
        assert torch.equal(run(k), whole[:k])


@pytest.mark.parametrize("E,N,K_,pairs,takes", [(1, 1, 256, 1, True), (512, 64, 256, 2048, True), (513, 64, 256, 8, False), (4, 64, 128, 8, False),
                                                (4, 64, 320, 8, False), (4, 64, 256, 2049, False)])
def test_what_all_waves_together_take(E, N, K_, pairs, takes):
    from braidinfer_amd import kernels as K
    assert bool(K._fn("experts_wide", "br_experts_wide_takes", [K.c_int] * 4)(E, N, K_, pairs)) == takes


@pytest.mark.parametrize("T,live", [(1, 1), (8, 6), (8, 0), (64, 40), (1024, 1000)])
def test_tokens_without_a_slot_go_to_no_expert(T, live):
    """Pairs of padding tokens are in nobody's run, and the outputs' sum leaves their rows as they are (or zero)."""
    from braidinfer_amd import kernels as K
    top, E, W = 3, 7, 20
    chosen = drawn(T, top, E, "drawn", T)
    g = torch.Generator().manual_seed(T + live)
    slots = torch.full((T,), -1, dtype=torch.int32)
    alive = torch.randperm(T, generator=g)[:live]
    slots[alive] = torch.arange(live, dtype=torch.int32)
    n = T * top
    first, order, place = (torch.full((k,), 9999, dtype=torch.int32, device="cuda") for k in (E + 1, n, n))
    K.experts_sort(chosen, first, order, place, E, slots=slots.cuda())
    c, first, order, place = chosen.cpu(), first.cpu(), order.cpu(), place.cpu().reshape(T, top)
    keep = slots >= 0
    assert first.tolist() == [int((c[keep] < e).sum()) for e in range(E + 1)]
    assert torch.all(place[~keep] == -1) and sorted(place[keep].reshape(-1).tolist()) == list(range(live * top))
    for t in alive.tolist():
        for s in range(top):
            assert int(order[place[t, s]]) == t * top + s and first[c[t, s]] <= place[t, s] < first[c[t, s] + 1]
    out = torch.full((n, W), float("nan"))
    out[:live * top] = torch.randn(live * top, W, generator=g)
    share, x = torch.rand(T, top, generator=g), torch.randn(T, W, generator=g)
    for store in (False, True):
        got = x.cuda()
        K.experts_combine(out.cuda(), place.reshape(-1).cuda(), share.cuda(), got, store=store)
        want = torch.zeros(T, W, dtype=torch.float64) if store else x.double()
        want[keep] += (share[keep][:, :, None].double() * out[place[keep].long()].double()).sum(1)
        assert (got.cpu().double() - want).abs().max() < 1e-5


@pytest.mark.parametrize("top", [1, 7, 8, 9, 17])
@pytest.mark.parametrize("W", [4, 1028, 30])
def test_combine_adds_every_slot(top, W):
    """Outputs asked for eight slots at a time: numbers of slots around that, widths with and without 16-byte reads."""
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(top)
    T = 5
    out, share, x = torch.randn(T * top, W, generator=g), torch.rand(T, top, generator=g), torch.randn(T, W, generator=g)
    place = torch.randperm(T * top, generator=g)
    terms = share[:, :, None].double() * out[place].reshape(T, top, W).double()
    for store in (False, True):
        got = x.cuda()
        K.experts_combine(out.cuda(), place.int().cuda(), share.cuda(), got, store=store)
        want = terms.sum(1) + (0 if store else x.double())
        assert ((got.cpu().double() - want).abs() <= (top + 1) * 2 ** -23 * (terms.abs().sum(1) + x.abs().double())).all()


@pytest.mark.parametrize("top", [1, 4, 5, 8])
@pytest.mark.parametrize("W,dtype", [(4, torch.bfloat16), (512, torch.float32), (1024, torch.bfloat16), (2044, torch.bfloat16),
                                     (2048, torch.bfloat16), (4096, torch.bfloat16), (4096, torch.float32)])
def test_combine_with_the_norm_behind_it(W, dtype, top):
    """The sum and the norm in one launch: the bits of the two, at widths around the workgroups' sizes; a token without outputs."""
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(top + W)
    T = 6
    out, share, x = (torch.randn(s, generator=g).cuda() for s in ((T * top, W), (T, top), (T, W)))
    place = torch.randperm(T * top, generator=g).int().reshape(T, top)
    place[2] = -1
    place, w = place.reshape(-1).cuda(), (1 + torch.randn(W, generator=g) / 4).cuda()
    assert K.experts_combine_norms(out, x, w)
    x2, y, y2 = x.clone(), torch.empty(T, W, dtype=dtype, device="cuda"), torch.empty(T, W, dtype=dtype, device="cuda")
    K.experts_combine(out, place, share, x)
    K.rmsnorm(x, w, y, 1e-5)
    K.experts_combine(out, place, share, x2, then=(w, 1e-5, y2))
    assert torch.equal(x, x2) and torch.equal(y, y2)


def test_combine_without_room_for_the_norm():
    from braidinfer_amd import kernels as K
    for W in (6, 2046, 4100, 8192):          # not in steps of 4, or beyond 16 floats a thread of 256
        assert not K.experts_combine_norms(torch.empty(2, W), torch.empty(2, W), torch.empty(W))


def test_rows_beyond_4_gb():
    """The second product of a step whose pairs' rows take more than 4 GB: the first and the last rows of every expert."""
    from braidinfer_amd import kernels as K
    Kd, N, n = 64, 16, 2 ** 25 + 700
    g = torch.Generator(device="cuda").manual_seed(1)
    starts = [0, 0, 300, 2 ** 25 - 131, 2 ** 25 + 200, n, n]
    E = len(starts) - 1
    first = torch.tensor(starts, dtype=torch.int32).cuda()
    w = torch.randn(E, N, Kd, device="cuda", generator=g).to(torch.bfloat16)
    a = torch.empty(n, Kd, dtype=torch.bfloat16, device="cuda")
    for i in range(0, n, 2 ** 22):
        a[i:i + 2 ** 22] = torch.randn(min(2 ** 22, n - i), Kd, device="cuda", generator=g)
    out = torch.full((n, N), 7.0, device="cuda")
    K.experts_gemm(a, w, first, out)
    for e in range(E):
        for lo, hi in {(starts[e], min(starts[e] + 400, starts[e + 1])), (max(starts[e], starts[e + 1] - 400), starts[e + 1])}:
            if hi > lo:
                want = a[lo:hi].double() @ w[e].double().T
                # float sums of 64 products: 64 2^-24 of the terms' sum, which is about 50
                assert float((out[lo:hi].double() - want).abs().max()) < 64 * 2 ** -24 * 50


# slots by counting (up to 16 experts, or 12 a slot for two slots and more) and by rounds of maxima
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (8, 32, 8), (16, 64, 64), (13, 63, 5), (5, 65, 3), (16, 512, 8), (9, 16, 1), (9, 17, 1), (7, 64, 1), (8, 24, 2),
                                     (8, 25, 2), (6, 48, 4), (6, 49, 4)])
def test_choice_and_sort_in_one_launch(T, E, top):
    """The same choice, shares and runs as by two launches, with equal scores, scores that are not numbers and infinite ones among
    them; the choice of finite scores is that of a stable sort, the shares its softmax."""
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(T + E)
    scores, bias = torch.randn(T, E, generator=g).mul(2).round(decimals=1), torch.randn(E, generator=g).round(decimals=1)
    wild = torch.zeros(T, dtype=torch.bool)
    if T > 4:
        scores[1, ::2], scores[2], scores[3, 0], scores[4, E // 2] = float("nan"), float("-inf"), float("inf"), float("-inf")
        wild[1:5] = True
    for b in (bias, None):
        bd, sd = (None if b is None else b.cuda()), scores.cuda()
        chosen, share = torch.full((T, top), -5, dtype=torch.int32, device="cuda"), torch.zeros(T, top, device="cuda")
        K.route_topk(sd, bd, chosen, share, top, 1.5)
        assert int(chosen.min()) >= 0 and int(chosen.max()) < E
        chosen2, share2 = torch.full_like(chosen, -5), torch.zeros_like(share)
        first, order, place = (torch.full((k,), 9999, dtype=torch.int32, device="cuda") for k in (E + 1, T * top, T * top))
        K.experts_sort(chosen2, first, order, place, E, route=(sd, bd, share2, 1.5))
        assert torch.equal(chosen, chosen2) and torch.equal(share.view(torch.int32), share2.view(torch.int32))
        c = chosen.cpu().reshape(-1)
        assert first.tolist() == [int((c < e).sum()) for e in range(E + 1)]
        assert torch.equal(order.cpu()[place.cpu().long()], torch.arange(T * top, dtype=torch.int32))
        assert all(int(first[e]) <= int(p) < int(first[e + 1]) for e, p in zip(c.tolist(), place.tolist()))
        z = (scores if b is None else scores + b)[~wild]
        v, at = torch.sort(z, dim=1, descending=True, stable=True)
        assert torch.equal(chosen.cpu()[~wild].long(), at[:, :top])
        want = 1.5 * torch.softmax(v[:, :top].double(), 1)
        assert float((share.cpu()[~wild].double() - want).abs().max()) < 1.5 * (top + 8) * 2 ** -24
