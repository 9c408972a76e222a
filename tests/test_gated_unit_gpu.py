"""The gated unit of the bfloat16 products over the gates whose sigmoid is below the smallest normal float and whose result is not."""
import pytest
import torch

import braidinfer_amd.kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows that go to the streaming kernels, the resident ones, the tiles of eight and of four waves; the experts' kernels of few and of many pairs
@pytest.mark.parametrize("M", [1, 16, 17, 64, 67, 96, 128, 129, 400])
@pytest.mark.parametrize("experts", [False, True])
def test_gates_far_below_zero(M, experts):
    Kd, I = 1024, 256
    gates = torch.cat([torch.arange(-88.5, -80.0, 0.5), torch.arange(-80.0, 81.0, 0.75), torch.tensor([-88.0, 100.0, 0.0])])[:I]
    gates = torch.nn.functional.pad(gates, (0, I - len(gates)), value=-87.5).to(DEV).bfloat16().float()
    wg, wu = (torch.zeros(I, Kd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    wg[:, 0], wu[:, 0] = gates, 1.0                       # every sum is one product: the gates as they are
    a = torch.zeros(M, Kd, device=DEV, dtype=torch.bfloat16)
    a[:, 0] = 1.0
    out = torch.empty(M, I, device=DEV, dtype=torch.bfloat16)
    if experts:
        first = torch.tensor([0, M], dtype=torch.int32, device=DEV)
        K.experts_up_tiles(a, torch.cat([wg, wu])[None], first, torch.arange(M, dtype=torch.int32, device=DEV), out, 1)
    else:
        scratch = torch.empty(K.GEMM_SCRATCH_FLOATS, device=DEV)
        K.gemm_swiglu(a, K.interleave_gate_up(wg, wu), out, scratch=scratch)
    g = gates.double()
    want = g / (1 + torch.exp(-g))
    # float operations and one rounding to the 8 bits of bfloat16
    assert ((out.double() - want).abs() <= (2 ** -8 + 2 ** -20) * want.abs()).all()
