"""Products of 65 to 96 rows by the resident workgroups that share the activations, against float64 and beside the tiles of eight waves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# both numbers of row blocks at their edges; weight rows that end in the middle of a tile and of a block of 16; two chunks of k and an odd number; every epilogue
@pytest.mark.parametrize("M", [65, 80, 81, 96])
@pytest.mark.parametrize("N,K_", [(16400, 256), (1000, 640), (70, 4096), (2048, 1408)])
@pytest.mark.parametrize("kind", ["bf16", "f32", "acc", "swiglu"])
def test_rows_of_five_and_six_blocks(M, N, K_, kind):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + N)
    if kind == "swiglu":
        N = -(-N // 16) * 16
    a = torch.randn(M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(N, K_, generator=g, device="cuda").mul(K_ ** -0.5).to(torch.bfloat16)
    want = a.double() @ w.double().T
    scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device="cuda")
    wide = torch.full((M + 1, (N // 2 if kind == "swiglu" else N) + 8), 7.0, device="cuda", dtype=torch.bfloat16 if kind in ("bf16", "swiglu") else torch.float32)
    out = wide[:M, :wide.shape[1] - 8]
    for kernel in (8, 8 + 16 * (4 + 16), 8 + 16 * (7 + 16)):       # as shaped, tiles of 64 and of 112 weight rows in one run
        out.fill_(7.0)
        if kind == "swiglu":
            K.gemm_swiglu(a, w, out, kernel=kernel, scratch=scratch)
            gate, up = (want.reshape(M, -1, 2, 8)[:, :, i].reshape(M, -1) for i in range(2))
            exact, bound = gate * torch.sigmoid(gate) * up, 2 ** -8
        else:
            K.gemm(a, w, out, accumulate=kind == "acc", kernel=kernel, scratch=scratch)
            exact, bound = want + (7.0 if kind == "acc" else 0.0), 2 ** -8 if kind == "bf16" else 4e-7
        assert float((out.double() - exact).norm() / exact.norm()) < bound
        assert bool((wide[M:] == 7.0).all()) and bool((wide[:, wide.shape[1] - 8:] == 7.0).all())
