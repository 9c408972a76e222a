"""Several products of few rows in one launch, against float64 products branch by branch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows at the edges of the kernels' 8, 16, 32 and 64; one branch and several; with 128 weight rows a branch (more compute units than
# tiles) and 16,384 (more tiles than compute units); an odd number of 128-wide chunks; a gap in front, between, behind and none
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("B,per,K_,gap_at,gap", [(4, 128, 1024, 3, 128), (1, 256, 1152, 0, 5), (3, 384, 1024, 3, 7), (2, 16384, 1152, 1, 16), (4, 2048, 2048, 0, 0)])
def test_branches(M, B, per, K_, gap_at, gap):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + per)
    a = torch.randn(B, M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(B * per, K_, generator=g, device="cuda").to(torch.bfloat16)
    wide = torch.full((M, B * per + gap + 4), 7.0, device="cuda")
    out = wide[:, :B * per + gap]
    K.gemm_branches(a, w, out, gap_at=gap_at, gap=gap)
    cols = torch.arange(B * per, device="cuda")
    cols = cols + gap * (cols >= gap_at * per)
    want = torch.cat([a[b].double() @ w[b * per:(b + 1) * per].double().T for b in range(B)], 1)
    assert float((out[:, cols].double() - want).norm() / want.norm()) < 4e-7        # float sums of K products
    left = torch.ones(wide.shape[1], dtype=torch.bool, device="cuda")
    left[cols] = False
    assert torch.all(wide[:, left] == 7.0)


# more than 128 rows: the last tile of one row, whole tiles, tiles cut short; columns of tiles behind, in front of and without a gap; one
# k-tile and more; more tiles than compute units; both tile heights
@pytest.mark.parametrize("M", [129, 255, 257, 449, 1024])
@pytest.mark.parametrize("B,per,K_,gap_at,gap", [(4, 256, 64, 3, 256), (2, 512, 192, 0, 4), (3, 256, 1024, 2, 12), (4, 2048, 512, 0, 0), (8, 4096, 128, 7, 8)])
def test_branches_of_many_rows(M, B, per, K_, gap_at, gap):
    from braidinfer_amd import kernels as K
    assert K.gemm_branches_pay(M, B, per, K_)
    test_branches(M, B, per, K_, gap_at, gap)
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn(B, M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(B * per, K_, generator=g, device="cuda").to(torch.bfloat16)
    out, again = (torch.empty(M, B * per, device="cuda") for _ in range(2))
    K.gemm_branches(a, w, out)
    K.gemm_branches(a.flip(0).contiguous(), torch.cat(w.split(per)[::-1]), again)      # a branch's bits do not depend on its place
    assert torch.equal(torch.cat(again.split(per, 1)[::-1], 1), out)


# eight, four, two runs along k and none; rows that end inside a tile; a last run that is shorter (K = 1,344: 22 k-tiles in runs of 6)
@pytest.mark.parametrize("M", [129, 130, 300, 512, 700, 1024])
@pytest.mark.parametrize("B,per,K_", [(4, 4096, 4096), (4, 2048, 2048), (2, 512, 1344), (3, 256, 1024)])
def test_branches_have_the_bits_of_the_products_one_by_one(M, B, per, K_):
    from braidinfer_amd import kernels as K
    room = K.GEMM_SCRATCH_FLOATS
    assert K.gemm_branches_pay(M, B, per, K_, room)
    g = torch.Generator(device="cuda").manual_seed(M + K_)
    a = torch.randn(B, M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(B * per, K_, generator=g, device="cuda").to(torch.bfloat16)
    scratch = torch.full((room,), float("nan"), device="cuda")
    want, out = torch.empty(M, B * per, device="cuda"), torch.full((M, B * per + 8), 7.0, device="cuda")
    for b in range(B):
        K.gemm(a[b], w[b * per:(b + 1) * per], want[:, b * per:(b + 1) * per], scratch=scratch)
    K.gemm_branches(a, w, out, gap_at=1, gap=8, room=room)
    assert torch.equal(out[:, :per], want[:, :per]) and torch.equal(out[:, per + 8:], want[:, per:])
    assert torch.all(out[:, per:per + 8] == 7.0)


def test_branches_beyond_32_bit_offsets_go_one_by_one():
    """What is said to pay is taken: rows and weights below 4 GB, as the tiles of four waves reach them."""
    from braidinfer_amd import kernels as K
    assert K.gemm_branches_pay(524287, 4, 4096, 4096) and not K.gemm_branches_pay(524288, 4, 4096, 4096)
    assert K.gemm_branches_pay(1801, 63, 8192, 4096) and not K.gemm_branches_pay(1801, 64, 8192, 4096)


def test_branches_of_many_rows_refuse():
    from braidinfer_amd import kernels as K
    from braidinfer_amd.errors import KernelError
    for M, B, per, K_ in ((128, 4, 256, 1024), (129, 1, 256, 1024), (129, 4, 384, 1024), (129, 4, 256, 1056)):
        assert not K.gemm_branches_pay(M, B, per, K_)
    a, w = torch.zeros(2, 129, 64, dtype=torch.bfloat16, device="cuda"), torch.zeros(512, 64, dtype=torch.bfloat16, device="cuda")
    for out in (torch.zeros(129, 515, device="cuda"), torch.zeros(129, 516, device="cuda")[:, 1:514]):
        with pytest.raises(KernelError):
            K.gemm_branches(a, w, out, gap_at=1, gap=out.shape[1] - 512)


def test_branches_refuse():
    from braidinfer_amd import kernels as K
    from braidinfer_amd.errors import KernelError
    for M, per, K_ in ((65, 128, 1024), (4, 64, 1024), (4, 128, 896), (4, 128, 1088)):
        assert not K.gemm_branches_takes(M, per, K_)
        a, w = torch.zeros(2, M, K_, dtype=torch.bfloat16, device="cuda"), torch.zeros(2 * per, K_, dtype=torch.bfloat16, device="cuda")
        with pytest.raises(KernelError):
            K.gemm_branches(a, w, torch.zeros(M, 2 * per, device="cuda"))


# one more branch whose sums' tanh goes to rows of its own: rows of one block, whole; few and many tiles; a tail of one tile, of several, as long as a branch
@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("B,per,K_,R,gap", [(4, 128, 1024, 16, 128), (1, 256, 1152, 256, 0), (4, 2048, 2048, 64, 2048), (2, 8192, 1024, 48, 3)])
def test_a_tail(M, B, per, K_, R, gap):
    from braidinfer_amd import kernels as K
    from braidinfer_amd.errors import KernelError
    g = torch.Generator(device="cuda").manual_seed(M + per)
    a = torch.randn(B + 1, M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(B * per + R, K_, generator=g, device="cuda").mul(K_ ** -0.5).to(torch.bfloat16)
    wide = torch.full((M, B * per + gap), 7.0, device="cuda")
    room = torch.full((M + 1, R), 7.0, device="cuda", dtype=torch.bfloat16)
    K.gemm_branches(a, w, wide, gap_at=B - 1, gap=gap, tail=room[:M])
    plain = torch.full_like(wide, 7.0)
    for b in range(B):                                   # (each branch as a product of its own)
        at = b * per + (gap if b == B - 1 else 0)
        K.gemm(a[b], w[b * per:(b + 1) * per], plain[:, at:at + per])
    assert float((wide - plain).norm() / plain.norm()) < 4e-7
    want = torch.tanh(a[B].double() @ w[B * per:].double().T)
    assert float((room[:M].double() - want).norm() / want.norm()) < 2 ** -8
    assert bool((room[M:] == 7.0).all())
    with pytest.raises(KernelError):
        K.gemm_branches(torch.cat([a] * 17, 1)[:, :17], w, torch.zeros(17, B * per, device="cuda"), tail=torch.zeros(17, R, device="cuda", dtype=torch.bfloat16))
