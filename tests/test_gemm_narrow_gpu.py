"""Products against at most 64 weight rows, at the edges of their blocks of 16 rows and chunks of 128 along k, against float64."""
import pytest
import torch

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
