"""The prompt products' tiles of four waves in products of more than one round of workgroups, whose last tiles multiply only the blocks that hold
rows, and of one round, whose last tiles multiply all: the bits of whole tiles."""
import pytest
import torch

import braidinfer_amd.kernels as K

pytestmark = pytest.mark.gpu


# blocks of 32 rows a wave in the last tile: one to four; 260 to 350 columns of tiles, the last of 20 weight rows, and one round of them
@pytest.mark.parametrize("kernel", [12, 13, 14, 15])
@pytest.mark.parametrize("M", [1, 64, 65, 129, 192, 193, 257, 320, 449])
@pytest.mark.parametrize("N", [66580, 1044])
def test_last_rows(kernel, M, N):
    Kd = 128
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(512, Kd, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, Kd, generator=g, device="cuda").mul(0.3).bfloat16()
    for dtype, accumulate in ((torch.bfloat16, False), (torch.float32, False), (torch.float32, True)):
        whole, got = torch.full((512, N), 0.25, device="cuda", dtype=dtype), torch.full((M + 1, N), 0.25, device="cuda", dtype=dtype)
        K.gemm(a, w, whole, accumulate=accumulate, kernel=kernel)
        K.gemm(a[:M], w, got[:M], accumulate=accumulate, kernel=kernel)
        assert torch.equal(got[:M], whole[:M]) and (got[M] == 0.25).all()
    want = a[:M].double() @ w.double().t() + 0.25
    assert (got[:M].double() - want).abs().max() <= want.abs().max() * 2e-6          # 128 products added in float
