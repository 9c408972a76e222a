"""Routed experts by the tiles of 128 and of 256 rows: both give every pair of every expert the same bits, which are right, wherever the
experts' rows end and however the columns of tiles are cut into runs."""
import pytest
import torch

import braidinfer_amd.kernels as K
from braidinfer_amd.errors import KernelError

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


# every number of blocks of a last tile of either height, alone and behind whole tiles; experts without rows; more than 64 experts; a last column
# of tiles of 16, 64 and 128 weight rows, one to nine of them; one k-tile, an odd number, and more
@pytest.mark.parametrize("counts", [[1], [64], [65], [130], [200], [256], [257, 0, 513], [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256], [0, 0, 700, 3, 0, 320],
                                    [450] * 16, [(i * 37) % 300 for i in range(70)]])
@pytest.mark.parametrize("W,F,N", [(64, 64, 16), (192, 576, 1088), (512, 1088, 576)])
def test_both_heights(counts, W, F, N):
    E, n = len(counts), sum(counts)
    h, gu, down = rnd(n, W, seed=n), rnd(E, 2 * F, W, seed=1, scale=W ** -0.5), rnd(E, N, F, seed=2, scale=F ** -0.5)
    first = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    order = torch.randperm(n, generator=torch.Generator().manual_seed(n)).to(torch.int32).to(DEV)
    a = rnd(n, F, seed=3)
    ups, downs = [], []
    for rows in (128, 256, 0):
        ups.append(torch.full((n + 1, F), float("nan"), device=DEV, dtype=torch.bfloat16))
        K.experts_up_tiles(h, gu, first, order, ups[-1][:n], 1, rows=rows)
        for dtype in (torch.float32, torch.bfloat16):
            downs.append(torch.full((n + 1, N), float("nan"), device=DEV, dtype=dtype))
            K.experts_gemm(a, down, first, downs[-1][:n], rows=rows)
    for y in ups:
        assert torch.equal(y[:n], ups[0][:n]) and y[n].isnan().all()
    for i, out in enumerate(downs):
        assert torch.equal(out[:n], downs[i % 2][:n]) and out[n].isnan().all()
    for e, c in enumerate(counts):
        if not c:
            continue
        at = slice(int(first[e]), int(first[e + 1]))
        s = h[order[at].long()].double() @ gu[e].double().t()
        want = s[:, :F] * torch.sigmoid(s[:, :F]) * s[:, F:]
        assert ((ups[0][at].double() - want).abs() <= 2 ** -8 * want.abs() + 1e-4).all()       # one rounding to bfloat16 of float sums
        want = a[at].double() @ down[e].double().t()
        assert (downs[0][at].double() - want).abs().max() <= 2e-6 * want.abs().max()           # float sums
        assert (downs[1][at].double() - want).abs().max() <= (2 ** -8 + 2e-6) * want.abs().max()


def test_heights_that_are_not_there():
    first = torch.tensor([0, 4], dtype=torch.int32, device=DEV)
    with pytest.raises(KernelError):
        K.experts_gemm(rnd(4, 64, seed=1), rnd(1, 16, 64, seed=2), first, torch.empty(4, 16, device=DEV), rows=64)


# 32 experts of 1,792 by 4,096, 16 of 1,408 by 2,048 and 8 of 2,048 by 1,024: pairs an expert where equal rows and uneven ones are faster by the height named, or as fast
@pytest.mark.parametrize("E,N,gated,tall,flat", [(32, 3584, True, (136, 150, 160, 400, 475, 512, 603, 675, 1800), (64, 96, 300, 350)),
                                                 (16, 2816, True, (136, 150, 160, 900, 1200), (64, 96, 300, 350, 400, 450, 475, 768)),
                                                 (32, 4096, False, (150, 200, 400, 603, 1800), (64, 128)), (16, 2048, False, (300, 350, 768, 1200, 1800), (64, 160, 603)),
                                                 (8, 1024, False, (1100,), (400, 768))])
def test_the_height_that_is_chosen(E, N, gated, tall, flat):
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    assert [K.experts_tiles_rows(m * E, E, N, gated) for m in tall] == [256] * len(tall)
    assert [K.experts_tiles_rows(m * E, E, N, gated) for m in flat] == [128] * len(flat)
