"""Products against at most 64 weight rows, at the edges of their blocks of 16 rows and chunks of 128 along k, against float64."""
import pytest
import torch

from braidinfer_amd.errors import KernelError

pytestmark = pytest.mark.gpu


# rows around one block of 16 and where a workgroup takes 1, 2 or 4 blocks of weight rows; K of whole chunks for every wave, of
# fewer chunks than waves, and cut short inside a chunk
@pytest.mark.parametrize("M", [17, 32, 33, 1801, 5003])
@pytest.mark.parametrize("N,K_", [(1, 4096), (16, 256), (17, 2048), (33, 264), (48, 4104), (64, 4096), (64, 1000)])
def test_few_weight_rows(M, N, K_):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + N + K_)
    wide = torch.randn(M, K_ + 8, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(N, K_, generator=g, device="cuda").to(torch.bfloat16)
    for a in (wide[:, :K_], wide[:, :K_].contiguous()):                  # rows that lie further apart, and dense ones
        want = a.double() @ w.double().T
        out = torch.full((M, N + 3), 7.0, device="cuda")
        K.gemm(a, w, out[:, :N])
        # float sums: at most K / 8 terms one after the other in a wave's chain, each rounding 2^-24 of the sum so far
        assert float((out[:, :N].double() - want).norm() / want.norm()) < 4e-7
        assert torch.all(out[:, N:] == 7.0)
        K.gemm(a, w, out[:, :N], accumulate=True)
        assert float((out[:, :N].double() - 2 * want).norm() / want.norm()) < 1e-6
        rounded = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        K.gemm(a, w, rounded)
        assert float((rounded.double() - want).norm() / want.norm()) < 2 ** -8


# every block width by force, beyond the sizes where it is chosen: rows of one block to many, K of one wave's chunk to several rounds of
# all waves' and cut short inside a chunk
@pytest.mark.parametrize("blocks", [1, 2, 4])
@pytest.mark.parametrize("M,N,K_", [(1, 1, 8), (16, 64, 128), (17, 33, 14336), (65, 64, 8200), (300, 80, 4096), (40, 16, 2056)])
def test_forced_blocks(blocks, M, N, K_):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + N + K_)
    a, w = torch.randn(M, K_, generator=g, device="cuda").to(torch.bfloat16), torch.randn(N, K_, generator=g, device="cuda").to(torch.bfloat16)
    want = a.double() @ w.double().T
    wide = torch.full((M, N + 3), 7.0, device="cuda")
    out = wide[:, :N]
    K.gemm(a, w, out, kernel=1 + 16 * blocks)
    assert float((out.double() - want).norm() / want.norm()) < 4e-7        # as above
    assert torch.all(wide[:, N:] == 7.0)
    with pytest.raises(KernelError):
        K.gemm(a, w, out, kernel=1 + 16 * 3)


# where a cut along k takes over: the last K of the narrow kernel for these rows, and the first beyond it
@pytest.mark.parametrize("M,last,beyond", [(65, 7168, 7232), (1024, 7168, 7232), (1025, 3072, 3136), (3072, 3072, 3136), (3073, 0, 256)])
def test_long_products_with_scratch_are_cut(M, last, beyond):
    from braidinfer_amd import kernels as K
    for N in (1, 32, 64):
        assert K.gemm_tile_choice(M, N, beyond, 1, K.GEMM_SCRATCH_FLOATS)[0] != 1
        assert not last or K.gemm_tile_choice(M, N, last, 1, K.GEMM_SCRATCH_FLOATS)[0] == 1
        assert K.gemm_tile_choice(M, N, beyond, 1, 0)[0] == 1 and K.gemm_tile_choice(M, 65, last or beyond, 1, 0)[0] != 1


# 17 to 64 rows: the runs that are left to a consumer are those of the product, or none
@pytest.mark.parametrize("M,N,K_,cut", [(17, 64, 3584, False), (32, 48, 3712, True), (33, 64, 4608, False), (64, 16, 4736, True), (17, 80, 2048, True)])
def test_runs_where_the_product_has_them(M, N, K_, cut):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M)
    a, w = torch.randn(M, K_, generator=g, device="cuda").to(torch.bfloat16), torch.randn(N, K_, generator=g, device="cuda").to(torch.bfloat16)
    scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device="cuda")
    want = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    K.gemm(a, w, want, scratch=scratch)
    runs = K.gemm_wide_partial(a, w, N, scratch)
    assert (runs > 1) == cut == (K.gemm_wide_parts(M, N, K_, scratch.numel(), accumulate=False) > 1)
    if cut:
        total = scratch[:M * N].clone()
        for r in range(1, runs):
            total += scratch[r * M * N:(r + 1) * M * N]
        assert torch.equal(total.reshape(M, N).to(torch.bfloat16), want)
