"""A product cut along k whose sum kernel also norms the rows: the rows of the two launches it stands for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows around the eight-wave tiles' 128 and at the ends of the range; columns of one to eight pieces of 1,024, whole and cut short
@pytest.mark.parametrize("M", [65, 128, 129, 300, 1024])
@pytest.mark.parametrize("N,K_,blocked", [(256, 4096, False), (1028, 2048, False), (2048, 1408, False), (4096, 4096, True), (5120, 2048, False),
                                          (8192, 1024, False)])
def test_sum_and_norm(M, N, K_, blocked):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(N, K_, generator=g, device="cuda").mul(K_ ** -0.5).to(torch.bfloat16)
    x, gain = torch.randn(M, N, generator=g, device="cuda"), torch.rand(N, generator=g, device="cuda") + 0.5
    scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device="cuda")
    if blocked:
        w = K.block_weight(w)
    want, want_h = x.clone(), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    K.gemm(a, w, want, accumulate=True, scratch=scratch)
    K.rmsnorm(want, gain, want_h, 1e-5)
    got, h = x.clone(), torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    runs = K.gemm_leave_runs(a, w, N, scratch)
    did = runs > 0
    _, parts, n1 = K.gemm_tile_choice(M, N, K_, mode=2, scratch_floats=scratch.numel())
    assert did == (parts > 1 and n1 == 0) and (not did or 2 <= runs <= parts)
    if not did:
        return
    K.rmsnorm(got, gain, h, 1e-5, add=(scratch, runs))
    assert torch.equal(got, want)
    # the sums of squares may be added in another order: a bfloat16 step (2^-8) of single elements at most
    assert float((h.float() - want_h.float()).abs().max()) <= 2 ** -8 * float(want_h.float().abs().max())
    assert float((h.float() - want_h.float()).norm() / want_h.float().norm()) < 1e-4


def test_refusals():
    from braidinfer_amd import kernels as K
    scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device="cuda")
    for M, N, K_ in ((64, 4096, 4096), (1025, 4096, 4096), (100, 8196, 1024), (100, 4096, 1000), (100, 64, 1024)):
        a, w = torch.zeros(M, K_, dtype=torch.bfloat16, device="cuda"), torch.zeros(N, K_, dtype=torch.bfloat16, device="cuda")
        assert K.gemm_leave_runs(a, w, N, scratch) == 0
