"""Products of 65 to 128 rows: what `gemm_tile_choice` names is what runs, bit for bit, for both layouts of the weights."""
import pytest
import torch

import braidinfer_amd.kernels as K
from braidinfer_amd.errors import KernelError

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M", [65, 67, 80, 81, 96, 128])
@pytest.mark.parametrize("N,Kd,mode", [(28672, 4096, 3), (17920, 4096, 3), (11264, 2048, 3), (16384, 4096, 0), (12288, 4096, 0), (32768, 4096, 1), (4096, 14336, 2)])
def test_the_choice_is_what_runs(M, N, Kd, mode):
    kernel, parts, n1 = K.gemm_tile_choice(M, N, Kd, mode, K.GEMM_SCRATCH_FLOATS)
    if kernel == 7:
        pytest.skip("rows of a workgroup are not named")
    assert n1 == 0 and kernel in (5, 6, 10)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(M, Kd, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, Kd, generator=g, device=DEV).mul(Kd ** -0.5).bfloat16()
    scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device=DEV)

    def run(weights, code):
        if mode == 3:
            out = torch.empty(M, N // 2, device=DEV, dtype=torch.bfloat16)
            K.gemm_swiglu(a, weights, out, kernel=code, scratch=scratch)
        else:
            out = torch.full((M, N), 0.25, device=DEV, dtype=torch.bfloat16 if mode == 0 else torch.float32)
            K.gemm(a, weights, out, accumulate=mode == 2, kernel=code, scratch=scratch)
        return out
    named = run(w, kernel + (16 * parts if parts > 1 else 0))
    assert torch.equal(run(w, 0), named)
    assert torch.equal(run(K.block_weight(w), 0), named)
    with pytest.raises(KernelError):                     # the resident workgroups take up to 64 rows
        run(w, 8)
