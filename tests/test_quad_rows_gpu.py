"""The prompt products' tiles of four waves where their rows or columns end: fewer blocks of rows in the last tile, rows written in runs
through LDS, and the experts' tiles in eight runs."""
import pytest
import torch

import braidinfer_amd.kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("kernel", [12, 13, 14, 15])
@pytest.mark.parametrize("M", [129, 192, 193, 256, 257, 320, 321, 448, 449])
def test_the_last_tile_has_the_bits_of_a_whole_one(kernel, M):
    N, Kd = 536, 192                                     # a last tile of columns that ends inside a run of 16 bytes' neighbours
    a, w = rnd(512, Kd, seed=M), rnd(N, Kd, seed=2, scale=0.3)
    for dtype, accumulate in ((torch.bfloat16, False), (torch.float32, False), (torch.float32, True)):
        wide = torch.full((512, N + 4), 0.25, device=DEV, dtype=dtype)            # rows of bfloat16 aligned to 8 bytes only
        K.gemm(a, w, wide[:, :N], accumulate=accumulate, kernel=kernel)
        got = torch.full((M + 1, N + 4), 0.25, device=DEV, dtype=dtype)
        K.gemm(a[:M], w, got[:M, :N], accumulate=accumulate, kernel=kernel)
        assert torch.equal(got[:M], wide[:M])
        assert (got[M] == 0.25).all() and (got[:, N:] == 0.25).all()              # nothing behind the last row or column
        want = a[:M].float() @ w.float().t() + (0.25 if accumulate else 0.0)
        # 192 products added in float, and one rounding of the result in bfloat16
        assert (got[:M, :N].float() - want).abs().max() <= want.abs().max() * (2 ** -8 if dtype == torch.bfloat16 else 2e-6)


@pytest.mark.parametrize("M", [130, 200, 321, 450])
def test_the_gated_unit_in_a_last_tile(M):
    I, Kd = 272, 256
    a = rnd(512, Kd, seed=M)
    wg, wu = rnd(I, Kd, seed=3, scale=0.3), rnd(I, Kd, seed=4, scale=0.3)
    w = K.interleave_gate_up(wg, wu)
    g, u = a.double() @ wg.double().t(), a.double() @ wu.double().t()
    want = g * torch.sigmoid(g) * u
    for kernel in (12, 13, 14, 15):
        whole, got = torch.empty(512, I, device=DEV, dtype=torch.bfloat16), torch.empty(M, I, device=DEV, dtype=torch.bfloat16)
        K.gemm_swiglu(a, w, whole, kernel=kernel)
        K.gemm_swiglu(a[:M], w, got, kernel=kernel)
        assert torch.equal(got, whole[:M])
        # one rounding to bfloat16 (2^-9) of float sums
        assert ((got.double() - want[:M]).abs() <= 2 ** -8 * want[:M].abs() + 1e-4).all()


@pytest.mark.parametrize("big", [1e3, 1e5, 3e38, float("inf")])
def test_the_gated_unit_at_the_ends_of_the_floats(big):
    """Gate values far out and infinite give what float arithmetic gives: the value times up, a zero, or no number."""
    Kd, M, I = 128, 160, 64
    a = torch.zeros(M, Kd, device=DEV, dtype=torch.bfloat16)
    a[:, 0] = 1.0
    wg = torch.zeros(I, Kd, device=DEV, dtype=torch.bfloat16)
    wu = torch.zeros_like(wg)
    wg[:, 0], wu[:, 0] = big, 0.5
    wg[1::2, 0] = -big
    wg[5, 0] = float("nan")
    out = torch.empty(M, I, device=DEV, dtype=torch.bfloat16)
    K.gemm_swiglu(a, K.interleave_gate_up(wg, wu), out, kernel=13)
    # (a zero times an infinite weight is no number: then every sum is none)
    g = (a.float() @ wg.float().t())[0] if big != float("inf") else wg[:, 0].float()
    want = (g / (1 + torch.exp(-g)) * 0.5).to(torch.bfloat16)
    assert torch.equal(torch.nan_to_num(out[7], nan=77.0), torch.nan_to_num(want, nan=77.0))


def counts(E, seed):
    g = torch.Generator().manual_seed(seed)
    edge = torch.tensor([0, 1, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 300, 513])
    return edge[torch.randint(0, len(edge), (E,), generator=g)].tolist()


@pytest.mark.parametrize("E,seed", [(1, 0), (3, 1), (8, 2), (32, 3), (64, 4), (70, 5)])
def test_every_pair_of_every_expert(E, seed):
    W, F, top = 128, 192, 2
    c = counts(E, seed)
    c[0] += 1 + (sum(c) + 1) % 2
    n = sum(c)
    T = n // top
    h, gu, down = rnd(T, W, seed=seed), rnd(E, 2 * F, W, seed=seed + 1, scale=0.3), rnd(E, W, F, seed=seed + 2, scale=0.3)
    first = torch.tensor([0] + torch.tensor(c).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    order = torch.randperm(n, generator=torch.Generator().manual_seed(seed)).to(torch.int32).to(DEV)
    y = torch.full((n + 1, F), float("nan"), device=DEV, dtype=torch.bfloat16)
    out = torch.full((n + 1, W), float("nan"), device=DEV, dtype=torch.float32)
    K.experts_up_tiles(h, gu, first, order, y[:n], top)
    K.experts_gemm(y[:n], down, first, out[:n])
    assert y[n].isnan().all() and out[n].isnan().all()
    for e in range(E):
        a, b = int(first[e]), int(first[e + 1])
        if a == b:
            continue
        s = h[(order[a:b] // top).long()].double() @ gu[e].double().t()
        want = s[:, :F] * torch.sigmoid(s[:, :F]) * s[:, F:]
        assert ((y[a:b].double() - want).abs() <= 2 ** -8 * want.abs() + 1e-4).all()
        want = y[a:b].double() @ down[e].double().t()
        assert (out[a:b].double() - want).abs().max() <= 2e-6 * want.abs().max()
