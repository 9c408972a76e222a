"""The 32-bit products at the edges of their kernels: every kernel gives an element the same bits, whatever the rows beside it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rnd(*shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g)


# k at 1, 7, 8, 9 and 30 whole 64s (segments that are empty, of one, of several); weight rows at and around 16 and 128
@pytest.mark.parametrize("N,Kd", [(1, 64), (15, 448), (16, 512), (17, 576), (127, 1920), (128, 512), (300, 1024), (4100, 576)])
def test_products_of_every_height(N, Kd):
    from braidinfer_amd import kernels as K
    a, w, base = rnd(300, Kd, seed=1), rnd(N, Kd, seed=2), rnd(300, N, seed=3)
    want = a.double() @ w.double().T
    scratch = torch.empty(8 * 300 * N, device="cuda")
    whole = None
    for M in (300, 1, 8, 9, 16, 17, 31, 33, 64, 81, 113, 128, 129):
        for room in (None, scratch):
            out = torch.full((M, N), 7.0, device="cuda")
            K.gemm(a[:M], w, out, scratch=room)
            if whole is None:
                whole = out
                # a float sum of K products in segments: well below the bound K 2^-24 |a| |w| of any order
                assert float((out.double() - want).abs().max()) < 4e-7 * Kd ** 0.5 * 6
            assert torch.equal(out, whole[:M])
            acc = base[:M].clone()
            K.gemm(a[:M], w, acc, accumulate=True, scratch=room)
            assert torch.equal(acc, base[:M] + whole[:M])


@pytest.mark.parametrize("M", [1, 3, 12, 40, 130])
def test_rows_that_lie_anywhere(M):
    """Rows of activations and results at any multiple of 4 bytes: the same bits as rows at multiples of 16."""
    from braidinfer_amd import kernels as K
    N, Kd = 130, 576
    a, w = rnd(M, Kd, seed=4), rnd(N, Kd, seed=5)
    want = torch.empty(M, N, device="cuda")
    K.gemm(a, w, want)
    for shift, more in ((1, 5), (2, 2), (0, 3)):
        wide_a, wide_o = torch.zeros(M, Kd + more + shift, device="cuda"), torch.full((M, N + more + shift), 7.0, device="cuda")
        wide_a[:, shift:shift + Kd] = a
        K.gemm(wide_a[:, shift:shift + Kd], w, wide_o[:, shift:shift + N])
        assert torch.equal(wide_o[:, shift:shift + N], want)
        assert torch.all(wide_o[:, :shift] == 7.0) and torch.all(wide_o[:, shift + N:] == 7.0)


# more tiles than two a compute unit: whole rounds, then segments in one run of columns, in several (a scratch that holds few), and in none
@pytest.mark.parametrize("M,N", [(40, 33000), (150, 20500), (320, 7001), (600, 4096)])
def test_whole_rounds_and_segments_behind_them(M, N):
    from braidinfer_amd import kernels as K
    Kd = 576
    a, w, base = rnd(M, Kd, seed=6), rnd(N, Kd, seed=7), rnd(M, N, seed=8)
    want = torch.empty(M, N, device="cuda")
    for r in range(0, M, 16):                             # 16 rows at a time: the streaming kernel
        K.gemm(a[r:r + 16], w, want[r:r + 16])
    for floats in (0, 8 * M * 64, 8 * M * 640, 8 * M * 4096 + 3, 8 * M * N):
        room = torch.empty(floats, device="cuda") if floats else None
        out = torch.full((M, N), 7.0, device="cuda")
        K.gemm(a, w, out, scratch=room)
        assert torch.equal(out, want)
        K.gemm(a, w, base.copy_(out), accumulate=True, scratch=room)
        assert torch.equal(base, want + want)
