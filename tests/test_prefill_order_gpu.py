"""Attention over prompts: whatever the order its workgroups are taken in, a sequence's rows are what they are alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu

I32 = dict(dtype=torch.int32, device="cuda")


# kv heads by the eight, half and a quarter of them, one, and numbers that do not divide eight; steps that are resident at once and not; equal lengths, sequences
# without most tiles, more sequences than are taken tile by tile
@pytest.mark.parametrize("nq,nkv,hd", [(32, 8, 128), (16, 4, 64), (8, 2, 128), (4, 1, 64), (12, 6, 64), (16, 16, 128)])
@pytest.mark.parametrize("lens", [[700], [500, 60], [33, 1, 257, 900], [90] * 16, [40 + 3 * (i % 5) for i in range(19)]])
def test_rows_do_not_depend_on_the_other_sequences(nq, nkv, hd, lens):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + nkv)
    pages = [-(-n // 64) for n in lens]
    order = torch.randperm(sum(pages), generator=g).tolist()
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    for b, n in enumerate(pages):
        for j in range(n):
            table[b, j] = order.pop()
    table = table.cuda()
    cache = torch.randn(sum(pages), 2, nkv, 64, hd, generator=g).bfloat16().cuda()
    q = torch.randn(sum(lens), nq * hd, generator=g).bfloat16().cuda()
    cu = [sum(lens[:b]) for b in range(len(lens) + 1)]

    def run(t0, t1, rows):
        out = torch.full((t1 - t0, nq * hd), 7.0, dtype=torch.bfloat16, device="cuda")
        K.attention_prefill_bf16(q[t0:t1], nq * hd, out, torch.tensor([cu[b] - t0 for b in rows] + [t1 - t0], **I32), torch.tensor(rows, **I32),
                                 torch.tensor([lens[b] for b in rows], **I32), table, cache, len(rows), max(lens[b] for b in rows), nq, nkv, hd, 64, None, hd ** -0.5)
        return out
    together = run(0, cu[-1], list(range(len(lens))))
    for b in range(len(lens)):
        assert torch.equal(run(cu[b], cu[b + 1], [b]), together[cu[b]:cu[b + 1]]), b
    assert torch.isfinite(together.float()).all()


@pytest.mark.parametrize("nq,nkv,dk,dv", [(16, 8, 128, 128), (8, 2, 128, 128), (6, 3, 128, 128), (32, 1, 256, 224), (16, 1, 192, 160)])
@pytest.mark.parametrize("lens", [[300, 40], [20, 270, 1, 130], [50] * 17])
def test_rows_of_the_windowed_kernel(nq, nkv, dk, dv, lens):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(sum(lens) + dk)
    pages = [-(-n // 64) for n in lens]
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages), generator=g).tolist()
    for b, n in enumerate(pages):
        for j in range(n):
            table[b, j] = order.pop()
    table = table.cuda()
    unit = torch.randn(sum(pages), nkv * 64 * (dk + dv), generator=g).bfloat16().cuda()
    q = torch.randn(sum(lens), nq * dk, generator=g).bfloat16().cuda()
    cu = [sum(lens[:b]) for b in range(len(lens) + 1)]

    def run(t0, t1, rows):
        out = torch.full((t1 - t0, nq * dv), 7.0, dtype=torch.bfloat16, device="cuda")
        K.pwa_prefill_bf16(q[t0:t1], out, torch.tensor([cu[b] - t0 for b in rows] + [t1 - t0], **I32), torch.tensor(rows, **I32),
                           torch.tensor([lens[b] for b in rows], **I32), table, unit, None, None, len(rows), 300, nq, nkv, dk, dv, 64, 100, 0, dk ** -0.5, False)
        return out
    together = run(0, cu[-1], list(range(len(lens))))
    for b in range(len(lens)):
        assert torch.equal(run(cu[b], cu[b + 1], [b]), together[cu[b]:cu[b + 1]]), b


# 2^24 workgroups and more in all: a launch may have 2^32 threads along each side of its grid
@pytest.mark.parametrize("nq,nkv,B,max_new", [(32, 8, 600, 131072), (8, 8, 2048, 131072)])
def test_many_sequences_and_a_long_one_allowed(nq, nkv, B, max_new):
    from braidinfer_amd import kernels as K
    hd = 64
    g = torch.Generator().manual_seed(B)
    lens = [1 + b % 3 for b in range(B)]
    cu = [0] + torch.tensor(lens).cumsum(0).tolist()
    cache = torch.randn(B, 2, nkv, 64, hd, generator=g).bfloat16().cuda()
    q = torch.randn(cu[-1], nq * hd, generator=g).bfloat16().cuda()
    args = (torch.tensor(cu, **I32), torch.arange(B, **I32), torch.tensor(lens, **I32), torch.arange(B, **I32)[:, None].contiguous(), cache, B)
    outs = []
    for longest in (3, max_new):
        outs.append(torch.full((cu[-1], nq * hd), 7.0, dtype=torch.bfloat16, device="cuda"))
        K.attention_prefill_bf16(q, nq * hd, outs[-1], *args, longest, nq, nkv, hd, 64, None, hd ** -0.5)
    assert torch.equal(outs[0], outs[1]) and torch.isfinite(outs[0].float()).all()
