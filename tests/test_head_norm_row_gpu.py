"""The norm of long rows kept in registers, against float64, at row lengths around its threads and registers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("e", [512, 516, 1028, 2044, 2048, 2052, 4096, 8192, 8196, 2049])
@pytest.mark.parametrize("gate,weight,sigmoid,first", [(False, False, False, False), (True, True, False, False), (True, True, True, True),
                                                       (True, False, False, True)])
def test_long_rows(dtype, e, gate, weight, sigmoid, first):
    from braidinfer_amd import kernels as K
    T, H, g = 3, 2, torch.Generator().manual_seed(e)
    o = torch.randn(T, H * e, generator=g)
    w = torch.rand(H * e, generator=g) + 0.5 if weight else None
    z = torch.randn(T, H * e, generator=g) if gate else None
    y = torch.empty(T, H * e, dtype=dtype, device="cuda")
    wide = torch.cat([torch.zeros(T, 4), z], 1).cuda()[:, 4:] if gate else None              # strided rows
    K.head_norm_gate(o.cuda(), w.cuda() if weight else None, wide, y, H, e, 1e-5, gate_sigmoid=sigmoid, gate_first=first)
    v = o.double().reshape(T, H, e)
    zz = None if z is None else (torch.sigmoid(z.double()) if sigmoid else torch.nn.functional.silu(z.double())).reshape(T, H, e)
    base = v * zz if first and gate else v
    want = v / torch.sqrt((base * base).mean(-1, keepdim=True) + 1e-5)
    if weight:
        want = want * w.double().reshape(H, e)
    if gate:
        want = want * zz
    # float: a few roundings each of 2^-24, and the sum's in the scale; bfloat16: its own rounding
    tol = 2 ** -19 if dtype == torch.float32 else 2 ** -8
    assert ((y.cpu().double().reshape(T, H, e) - want).abs() <= tol * want.abs() + 1e-7).all()
