"""Attention over prompts with keys and values brought by direct loads: the bits of the form that stages pages through registers (which
takes what has a longer list of pages), and plain attention in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
NO_WINDOW = 1 << 30


# the three pairs of widths; several kv heads, one for all; windows without and with pooled rows, runs of positions, kept tokens, bounded
# scores, two maps; first portions and later ones (`before` tokens in the cache), rows that end inside a tile, a wave, a block of 32 keys
@pytest.mark.parametrize("dk,dv,H,G", [(128, 128, 8, 2), (192, 160, 16, 1), (256, 224, 32, 1)])
@pytest.mark.parametrize("size,pool,chunk,keep,cap,maps", [(NO_WINDOW, 0, 0, 0, 0.0, 1), (70, 0, 0, 0, 0.0, 1), (96, 5, 0, 0, 0.0, 1), (NO_WINDOW, 0, 100, 0, 20.0, 1),
                                                           (64, 0, 0, 40, 0.0, 1), (200, 0, 0, 0, 0.0, 2)])
@pytest.mark.parametrize("lens,before", [((67, 1, 200), (0, 300, 0)), ((33, 129, 64), (500, 31, 64))])
def test_direct_loads_give_the_bits_of_staged_pages(dk, dv, H, G, size, pool, chunk, keep, cap, maps, lens, before):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(dk + size % 1000 + lens[0])
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    B, T, nq = len(lens), sum(lens), H * maps
    ctx = [a + b for a, b in zip(lens, before)]
    per, pper = max(ctx) // 64 + 1, max(ctx) // 64 + 1
    perm = torch.randperm(B * per + 3, generator=torch.Generator().manual_seed(1))
    table = perm[:B * per].reshape(B, per).to(torch.int32).cuda()
    ptable = torch.arange(B * pper).reshape(B, pper).to(torch.int32).cuda()
    unit = torch.full((B * per + 3, G * 64 * (maps * dk + dv)), float("nan"), device="cuda", dtype=torch.bfloat16)      # what is not written shows
    pooled = torch.full((B * pper, G * 64 * (dk + dv)), float("nan"), device="cuda", dtype=torch.bfloat16)
    keys, values = [], []
    for b in range(B):
        k, v = rnd(ctx[b], G, maps * dk).to(torch.bfloat16), rnd(ctx[b], G, dv).to(torch.bfloat16)
        keys.append(k), values.append(v)
        for p in range(ctx[b]):
            u = unit[table[b, p // 64]]
            u[:G * 64 * maps * dk].view(G, 64, maps * dk)[:, p % 64] = k[p]
            u[G * 64 * maps * dk:].view(G, dv, 64)[:, :, p % 64] = v[p]
        for r in range(ctx[b] // pool if pool else 0):
            u = pooled[ptable[b, r // 64]]
            u[:G * 64 * dk].view(G, 64, dk)[:, r % 64] = k[r * pool:(r + 1) * pool].float().mean(0).to(torch.bfloat16)
            u[G * 64 * dk:].view(G, dv, 64)[:, :, r % 64] = v[r * pool:(r + 1) * pool].float().mean(0).to(torch.bfloat16)
    q = rnd(T, nq * dk).to(torch.bfloat16)
    sinks = rnd(nq)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    slots, ctx_d = torch.arange(B, dtype=torch.int32, device="cuda"), torch.tensor(ctx, dtype=torch.int32, device="cuda")
    scale = dk ** -0.5
    if maps > 1 and pool:
        pytest.skip("no pooled rows with maps")

    def run(t):
        out = torch.empty(T, nq * dv, device="cuda", dtype=torch.bfloat16)
        K.pwa_prefill_bf16(q, out, cu, slots, ctx_d, t, unit, ptable if pool else None, pooled if pool else None, B, max(lens), nq, G, dk, dv, 64, size,
                           pool, scale, True, sinks, chunk, keep, cap, maps)
        return out
    got = run(table)
    wide = torch.zeros(B, 4000, dtype=torch.int32, device="cuda")
    wide[:, :per] = table
    assert torch.equal(got, run(wide))
    if (chunk, keep, cap, pool) == (0, 0, 0.0, 0):
        for b in range(B):
            at = torch.arange(before[b], ctx[b], device="cuda")[:, None]
            seen = (torch.arange(ctx[b], device="cuda")[None] <= at) & (torch.arange(ctx[b], device="cuda")[None] > at - size)
            qb = q[int(cu[b]):int(cu[b + 1])].double().view(lens[b], nq, dk)
            for h in range(nq):
                kv = h // maps // (H // G)
                s = qb[:, h] @ keys[b][:, kv, (h % maps) * dk:(h % maps + 1) * dk].double().t() * scale
                s = torch.where(seen, s, -torch.inf)
                top = s.max(1, keepdim=True).values.clamp(min=float(sinks[h]))
                e = (s - top).exp()
                want = e @ values[b][:, kv].double() / (e.sum(1, keepdim=True) + (sinks[h].double() - top).exp())
                o = got[int(cu[b]):int(cu[b + 1])].view(lens[b], nq, dv)[:, h].double()
                # weights and results rounded to bfloat16
                assert (o - want).abs().max() < 2 ** -7 * values[b].abs().max().double()
