"""attention_simple: a query alone (four waves, a class of key chunks each) and among many (one wave for all classes) gives the
same bits, at context lengths around the chunks and classes, with and without a window."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd,window", [(128, None), (128, 100), (48, None), (24, 70), (320, 300), (6, None)])
def test_alone_and_among_many(dtype, hd, window):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(hd)
    page, T, nq, nkv = 64, 600, 2, 1
    q, k, v = (torch.randn(T, n, hd, generator=g).to(dtype) for n in (nq, nkv, nkv))
    n_pages = -(-T // page)
    cache = torch.full((n_pages, 2, nkv, page, hd), float("nan"), dtype=dtype)        # rows not written are never read
    pages = torch.randperm(n_pages, generator=g).tolist()
    for t in range(T):
        cache[pages[t // page], 0, :, t % page] = k[t]
        cache[pages[t // page], 1].view(nkv, hd, page)[:, :, t % page] = v[t]
    cache, table = cache.cuda(), torch.tensor([pages], dtype=torch.int32).cuda()
    qd = q.reshape(T, nq * hd).cuda()
    pos = torch.arange(T, dtype=torch.int32).cuda()
    zeros, slots = torch.zeros(20000, dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()

    def run(rows):
        out = torch.empty(len(rows), nq * hd, dtype=dtype, device="cuda")
        K.attention_simple(qd[rows].contiguous(), nq * hd, out, pos[rows].contiguous(), zeros[:len(rows)], slots, table, cache, len(rows),
                           nq, nkv, hd, page, window, 1 / math.sqrt(hd))
        return out
    some = [0, 1, 62, 63, 64, 65, 127, 128, 191, 192, 255, 256, 257, 319, 320, 511, 512, 599]
    many = torch.arange(T).repeat(20)
    whole = run(many.cuda())
    for t in some:
        assert torch.equal(run(torch.tensor([t]).cuda())[0], whole[t])
    kd, vd = k[:, 0].double(), v[:, 0].double()
    for t in some:
        lo = 0 if window is None else max(0, t - window + 1)
        for h in range(nq):
            w = torch.softmax((kd[lo:t + 1] @ q[t, h].double()) / math.sqrt(hd), 0)
            want = w @ vd[lo:t + 1]
            tol = 2e-6 if dtype == torch.float32 else 2 ** -8
            assert float((whole[t, h * hd:(h + 1) * hd].double().cpu() - want).abs().max()) < tol * max(1.0, float(want.abs().max())) * 2


@pytest.mark.parametrize("keys", [(0, 64), (64, 128), (70, 90), (128, 192), (64, 320), (0, 320)])
@pytest.mark.parametrize("what", ["not a number", "minus infinity"])
def test_scores_that_are_not_finite(keys, what):
    """Keys whose scores are not numbers show in every query that sees them, whichever chunks and classes they fill; scores of
    minus infinity weigh nothing, unless there are no others.  A query alone and among many."""
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(2)
    page, T, hd = 64, 320, 32
    q, k, v = (torch.randn(T, hd, generator=g) for _ in range(3))
    q[:, 0] = q[:, 0].abs() + 0.1
    k[keys[0]:keys[1], 0] = float("nan") if what == "not a number" else float("-inf")
    cache = torch.zeros(T // page, 2, 1, page, hd)
    cache[:, 0, 0] = k.reshape(-1, page, hd)
    cache[:, 1, 0].view(-1, hd, page)[:] = v.reshape(-1, page, hd).transpose(1, 2)
    cache, table = cache.cuda(), torch.arange(T // page, dtype=torch.int32).reshape(1, -1).cuda()
    zeros, slots = torch.zeros(20000, dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    qd, pos = q.cuda(), torch.arange(T, dtype=torch.int32).cuda()

    def run(rows):
        out = torch.empty(len(rows), hd, device="cuda")
        K.attention_simple(qd[rows].contiguous(), hd, out, pos[rows].contiguous(), zeros[:len(rows)], slots, table, cache, len(rows),
                           1, 1, hd, page, None, 1 / math.sqrt(hd))
        return out.cpu()
    whole = run(torch.arange(T).repeat(40).cuda())[:T]
    for t in (0, 63, 64, 75, 127, 128, 200, 255, 256, 319):
        want = torch.softmax((k[:t + 1].double() @ q[t].double()) / math.sqrt(hd), 0) @ v[:t + 1].double()
        for got in (whole[t], run(torch.tensor([t]).cuda())[0]):
            assert torch.equal(got.isnan(), want.isnan())
            if not want.isnan().any():
                assert float((got.double() - want).abs().max()) < 4e-6 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd,window", [(128, 100), (64, 65), (40, 3), (72, 129), (128, None)])
def test_values_read_one_by_one_and_16_bytes_at_a_time(dtype, hd, window):
    """Pages of 32 tokens read values one by one, pages of 64 and 128 16 bytes at a time from wherever a window's chunks start: the
    same bits, for a query alone and among many."""
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(hd)
    T, nq, nkv = 384, 2, 1
    q, k, v = (torch.randn(T, n, hd, generator=g).to(dtype) for n in (nq, nkv, nkv))
    qd, pos = q.reshape(T, nq * hd).cuda(), torch.arange(T, dtype=torch.int32).cuda()
    zeros, slots = torch.zeros(20000, dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    some = torch.tensor([0, 1, 30, 63, 64, 99, 100, 101, 163, 200, 229, 383])
    got = []
    for page in (32, 64, 128):
        n = T // page
        pages = torch.randperm(n, generator=g)
        cache = torch.empty(n, 2, nkv, page, hd, dtype=dtype)
        cache[pages, 0, 0] = k[:, 0].reshape(n, page, hd)
        cache[pages, 1, 0] = v[:, 0].reshape(n, page, hd).transpose(1, 2).reshape(n, page, hd)        # channels of a page's keys
        cache, table = cache.cuda(), pages.int().reshape(1, -1).cuda()

        def run(rows):
            out = torch.empty(len(rows), nq * hd, dtype=dtype, device="cuda")
            K.attention_simple(qd[rows].contiguous(), nq * hd, out, pos[rows].contiguous(), zeros[:len(rows)], slots, table, cache, len(rows),
                               nq, nkv, hd, page, window, 1 / math.sqrt(hd))
            return out
        got += [run(torch.arange(T).repeat(20).cuda())[some], torch.cat([run(t[None].cuda()) for t in some])]
    assert all(torch.equal(x, got[0]) for x in got[1:])
