"""Single tokens on the matrix cores: a sequence alone (its value channels over several workgroups) and among many (fewer, down to
one workgroup for all) has the same bits, and agrees with float64, at widths around the blocks of 32 and the registers' limits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk,dv", [(128, 128), (256, 224), (256, 256), (136, 100), (96, 64), (64, 96), (72, 40), (8, 4), (128, 160), (40, 132)])
@pytest.mark.parametrize("window,keep,cap", [(1 << 30, 0, 0.0), (100, 9, 20.0)])
def test_alone_and_among_many(dk, dv, window, keep, cap):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(dk + dv)
    lens = [1, 31, 32, 33, 64, 65, 200, 333]
    nkv, G, page, n = 2, 4, 64, len(lens)
    nq, scale = nkv * G, dk ** -0.5
    assert K.pwa_decode_takes(torch.bfloat16, nq, nkv, dk, dv, page)
    ks = [torch.randn(L, nkv, dk, generator=g).bfloat16() for L in lens]
    vs = [torch.randn(L, nkv, dv, generator=g).bfloat16() for L in lens]
    pages = [-(-L // page) for L in lens]
    order = torch.randperm(sum(pages), generator=g).tolist()
    table = torch.zeros(n, max(pages), dtype=torch.int32)
    # what is not written holds NaN in the values (read as zero) and numbers in the keys (masked)
    keys = torch.ones(sum(pages), nkv, page, dk, dtype=torch.bfloat16)
    values = torch.full((sum(pages), nkv, dv, page), float("nan"), dtype=torch.bfloat16)
    for b in range(n):
        for j in range(pages[b]):
            at = table[b, j] = order.pop()
            part = slice(64 * j, min(64 * j + 64, lens[b]))
            w = part.stop - part.start
            keys[at, :, :w] = ks[b][part].transpose(0, 1)
            values[at, :, :, :w] = vs[b][part].permute(1, 2, 0)
    unit = torch.cat([keys.reshape(len(keys), -1), values.reshape(len(values), -1)], 1).cuda()
    q = torch.randn(n, nq * dk, generator=g).bfloat16()
    qd, table, ctx = q.cuda(), table.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()

    def run(rows):
        rows = torch.tensor(rows)
        out = torch.empty(len(rows), nq * dv, dtype=torch.bfloat16, device="cuda")
        K.pwa_decode_bf16(qd[rows.cuda()].contiguous(), out, rows.int().cuda(), ctx[rows.cuda()].contiguous(), table, unit, None, None, len(rows), nq,
                          nkv, dk, dv, page, window, 0, scale, False, keep=keep, softcap=cap)
        return out
    alone = torch.cat([run([b]) for b in range(n)])
    for times in (1, 5, 9, 17, 40):
        many = run(list(range(n)) * times).reshape(times, n, -1)
        assert all(torch.equal(many[i], alone) for i in range(times)), times
    for b, L in enumerate(lens):
        lo = max(0, L - window)
        seen = [t for t in range(L) if t >= lo or t < keep]
        for h in range(nq):
            s = ks[b][seen, h // G].double() @ q[b, h * dk:(h + 1) * dk].double() * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            v = vs[b][seen, h // G].double()
            w = torch.softmax(s, 0)
            # probabilities and result rounded to 8 bits, sums in float
            bound = 2 ** -8 * (w @ v.abs() + (w @ v).abs()) + 1e-3
            assert (alone[b, h * dv:(h + 1) * dv].double().cpu() - w @ v).abs().le(bound).all(), (L, h)
