"""Single-token attention whose workgroups make more than one and up to two rounds of the compute units: the second round takes the sequences
from the last on, and every sequence's row is what it is alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# sequences * kv heads * runs of 256 compute units: just beyond one round, two whole rounds, one more than those (as they come), and heads
# that do not divide the units (as they come)
@pytest.mark.parametrize("B,nkv,nsplit,hd", [(33, 8, 1, 128), (64, 8, 1, 128), (65, 8, 1, 128), (40, 8, 1, 64), (8, 8, 8, 128), (5, 8, 8, 64), (90, 3, 1, 128)])
def test_rows_do_not_depend_on_their_place(B, nkv, nsplit, hd):
    from braidinfer_amd import kernels as K
    g = torch.Generator().manual_seed(B + hd)
    G, page = 2, 64
    nq, scale = nkv * G, hd ** -0.5
    lens = [1 + (37 * b) % 300 for b in range(B)]
    pages = [-(-L // page) for L in lens]
    order = torch.randperm(sum(pages), generator=g).tolist()
    table = torch.zeros(B, max(pages), dtype=torch.int32)
    for b in range(B):
        for j in range(pages[b]):
            table[b, j] = order.pop()
    cache = torch.randn(sum(pages), 2, nkv, page, hd, generator=g).bfloat16().cuda()
    q = torch.randn(B, nq * hd, generator=g).bfloat16().cuda()
    table, slots, ctx = table.cuda(), torch.arange(B, dtype=torch.int32).cuda(), torch.tensor(lens, dtype=torch.int32).cuda()

    def run(rows):
        n = len(rows)
        out = torch.full((n, nq * hd), 7.0, dtype=torch.bfloat16, device="cuda")
        part_o, part_ml = torch.empty(n * nq * nsplit * hd, device="cuda"), torch.empty(n * nq * nsplit * 2, device="cuda")
        K.attention_decode_bf16(q[rows].contiguous(), nq * hd, out, slots[rows].contiguous(), ctx[rows].contiguous(), table, cache, n, nq, nkv, hd, page, None, scale,
                                nsplit, part_o, part_ml, 2)
        return out
    together = run(torch.arange(B).cuda())
    for rows in (torch.arange(B - 1, -1, -1).cuda(), torch.arange(0, B, 3).cuda(), torch.tensor([B - 1]).cuda()):
        assert torch.equal(run(rows), together[rows])
    assert torch.isfinite(together.float()).all()
