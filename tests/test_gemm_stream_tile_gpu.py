"""Products by workgroups that hold a tile of 16, 24 or 32 weight rows over the whole of K: against double sums, at the edges
of tiles, rows and chunks, and where the rule takes them."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def bound(K):
    """A chain of K / 32 additions, each rounded to 2^-24 of what it holds, errs like a random walk."""
    return 2.0 ** -24 * (K / 32) ** 0.5


def operands(M, N, K_, seed, blocked=False):
    from braidinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn(M, K_, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(N, K_, generator=g, device="cuda").mul(K_ ** -0.5).to(torch.bfloat16)
    return a, w, (K.block_weight(w) if blocked else w), a.double() @ w.double().T


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


# the last rows of a block and the first of the next; K of fewer chunks than waves, of odd shares, whole; N below, at and behind tiles
@pytest.mark.parametrize("rt", [16, 24, 32])
@pytest.mark.parametrize("M,N,K_", [(1, 16, 1024), (8, 100, 256), (16, 49, 1408), (17, 72, 384), (32, 96, 4096), (33, 25, 1024), (48, 200, 640),
                                    (64, 33, 2048), (65, 1000, 1024), (80, 31, 896), (96, 64, 256), (97, 130, 1152), (112, 24, 1024), (113, 90, 1024),
                                    (128, 260, 1280)])
def test_tiles(rt, M, N, K_):
    from braidinfer_amd import kernels as K
    code = 7 + 16 * (rt // 8 - 1)
    for blocked in (False, True) if K_ >= 1024 else (False,):
        a, _, w, want = operands(M, N, K_, M + N, blocked)
        room = torch.full((M, N + 11), 7.0, device="cuda")
        for lead in (0, 3):                              # rows that 16-byte stores take, and others
            out = room[:, lead:lead + N]
            room.fill_(7.0)
            K.gemm(a, w, out, kernel=code)
            assert off(out, want) < bound(K_)
            assert bool((room[:, :lead] == 7.0).all()) and bool((room[:, lead + N:] == 7.0).all())
        base = torch.randn(M, N, device="cuda")
        got = base.clone()
        K.gemm(a, w, got, accumulate=True, kernel=code)
        assert off(got, base.double() + want) < bound(K_)
        half = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        K.gemm(a, w, half, kernel=code)
        f32 = torch.empty(M, N, device="cuda")
        K.gemm(a, w, f32, kernel=code)
        assert torch.equal(half, f32.to(torch.bfloat16))
        wide = torch.randn(M, K_ + 24, device="cuda").to(torch.bfloat16)
        wide[:, 8:8 + K_] = a
        again = torch.empty_like(f32)
        K.gemm(wide[:, 8:8 + K_], w, again, kernel=code)
        assert torch.equal(again, f32)


# rows that are added to: four columns at once where they lie at 16 bytes, each by itself where not; the last block of a tile of 24 begins at its
# eighth row, and columns end in the middle of a tile
@pytest.mark.parametrize("rt", [16, 24, 32])
@pytest.mark.parametrize("M,N,K_", [(1, 16, 1024), (9, 100, 1024), (16, 72, 1024), (24, 44, 512), (33, 4104, 256), (64, 120, 1024), (97, 49, 1024), (128, 200, 640)])
def test_rows_added_to(rt, M, N, K_):
    from braidinfer_amd import kernels as K
    code = 7 + 16 * (rt // 8 - 1)
    a, _, w, _ = operands(M, N, K_, M + rt)
    f32 = torch.empty(M, N, device="cuda")
    K.gemm(a, w, f32, kernel=code)
    for lead in (0, 4, 3):
        room = torch.randn(M, N + 12 - N % 4, device="cuda")
        want = room.clone()
        want[:, lead:lead + N] += f32
        K.gemm(a, w, room[:, lead:lead + N], accumulate=True, kernel=code)
        assert torch.equal(room, want)


# the sum of a product's runs by one and by four columns a thread
@pytest.mark.parametrize("M,N,K_,parts", [(70, 2048, 1024, 4), (70, 2052, 1024, 4), (128, 1028, 2048, 8), (66, 3072, 640, 2)])
def test_sums_of_runs(M, N, K_, parts):
    from braidinfer_amd import kernels as K
    a, w, _, want = operands(M, N, K_, N)
    scratch = torch.full((parts * M * N,), float("nan"), device="cuda")
    for lead in (0, 1):
        room = torch.full((M, N + 4), 7.0, device="cuda")
        K.gemm(a, w, room[:, lead:lead + N], kernel=6 + 16 * parts, scratch=scratch)
        assert off(room[:, lead:lead + N], want) < bound(K_)
        assert bool((room[:, :lead] == 7.0).all()) and bool((room[:, lead + N:] == 7.0).all())
        base = torch.randn(M, N + 4, device="cuda")
        got = base.clone()
        K.gemm(a, w, got[:, lead:lead + N], accumulate=True, kernel=6 + 16 * parts, scratch=scratch)
        base[:, lead:lead + N] += room[:, lead:lead + N]
        assert torch.equal(got, base)
    half = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    K.gemm(a, w, half, kernel=6 + 16 * parts, scratch=scratch)
    assert torch.equal(half, room[:, 1:1 + N].to(torch.bfloat16))


@pytest.mark.parametrize("rt", [16, 32])
@pytest.mark.parametrize("M,I,K_", [(1, 8, 1024), (16, 264, 1024), (24, 40, 512), (50, 72, 1024), (64, 328, 2048), (90, 200, 1152), (128, 24, 1024)])
def test_gated_unit(rt, M, I, K_):
    from braidinfer_amd import kernels as K
    a, wg, _, g = operands(M, I, K_, 1)
    wu = torch.randn(I, K_, device="cuda").mul(K_ ** -0.5).to(torch.bfloat16)
    want = g / (1 + torch.exp(-g)) * (a.double() @ wu.double().T)
    room = torch.full((M, I + 5), 7.0, dtype=torch.bfloat16, device="cuda")
    for lead in (0, 1):
        out = room[:, lead:lead + I]
        K.gemm_swiglu(a, K.interleave_gate_up(wg, wu), out, kernel=7 + 16 * (rt // 8 - 1))
        assert off(out, want) < 2 ** -8                  # one rounding to bfloat16
        assert bool((room[:, lead + I:] == 7.0).all())
    with pytest.raises(Exception, match="gemm_swiglu"):  # gates and up values of a block lie in one tile
        K.gemm_swiglu(a, K.interleave_gate_up(wg, wu), out, kernel=7 + 16 * 2)


# (rows, width of the normed rows, inner width, width of the product that reads them): tiles of 16 and 32, sums of squares by 16 columns
# or, where the first product is cut along k (the last two), by 256; the second product of either kernel
@pytest.mark.parametrize("M,H,Kd,N2", [(1, 4096, 1024, 6144), (9, 8192, 1024, 48), (16, 1024, 4096, 4096), (17, 1024, 2048, 304), (33, 4096, 1024, 28672),
                                       (64, 2048, 1024, 5120), (64, 8192, 1024, 1040), (40, 4096, 14336, 6144), (64, 4096, 14336, 28672)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_a_norm_prepared_and_used(M, H, Kd, N2, swiglu):
    from braidinfer_amd import kernels as K
    a, _, w1, y = operands(M, H, Kd, M)
    x0 = torch.randn(M, H, device="cuda") * torch.logspace(-1, 1, M, device="cuda")[:, None]
    gain = 1.0 + 0.2 * torch.randn(H, device="cuda")
    w2 = torch.randn(N2, H, device="cuda").mul(H ** -0.5).to(torch.bfloat16)
    scratch = torch.full((K.GEMM_SCRATCH_FLOATS,), float("nan"), device="cuda")
    xg = torch.empty(M, H, dtype=torch.bfloat16, device="cuda")
    ssq = torch.full((H // 16 * K.SSQ_LD,), float("nan"), device="cuda")
    x = x0.clone()
    tiles = K.gemm_norm_prepare(a, w1, x, gain, xg, ssq, scratch, whole=True)
    assert tiles == (H // 16 if M <= 16 or K.gemm_whole_pays(M, H, Kd, by16=True) else H // 256)
    sum_ = x0.double() + y
    assert off(x, sum_) < bound(Kd)
    assert torch.equal(xg, (x * gain).to(torch.bfloat16))
    squares = ssq[:tiles * K.SSQ_LD].view(tiles, K.SSQ_LD)[:, :M].double().sum(0)
    assert float((squares / (x.double() ** 2).sum(1) - 1).abs().max()) < bound(H)
    want = (xg.double() @ w2.double().T) * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    if swiglu:
        out = torch.empty(M, N2 // 2, dtype=torch.bfloat16, device="cuda")
        K.gemm_norm_scaled(xg, ssq, tiles, 1e-5, w2, out, swiglu=True, scratch=scratch, whole=True)
        gu = want.view(M, N2 // 16, 2, 8)
        g, u = gu[:, :, 0].reshape(M, -1), gu[:, :, 1].reshape(M, -1)
        assert off(out, g / (1 + torch.exp(-g)) * u) < 2 ** -8
    else:
        out = torch.empty(M, N2, device="cuda")
        K.gemm_norm_scaled(xg, ssq, tiles, 1e-5, w2, out, scratch=scratch, whole=True)
        assert off(out, want) < bound(H)


# widths that end in the middle of a tile of 32: nothing is written behind the last column, row or tile of squares
@pytest.mark.parametrize("M", [1, 8, 16, 24, 64])
@pytest.mark.parametrize("H", [4112, 5200, 8176])
def test_a_norm_prepared_up_to_the_last_column(M, H):
    from braidinfer_amd import kernels as K
    a, _, w, y = operands(M, H, 1024, M)
    x0, gain = torch.randn(M, H, device="cuda"), 1.0 + 0.2 * torch.randn(H, device="cuda")
    P, I, Z = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t
    prepare = K._fn("gemm_bf16", "br_gemm_bf16_norm_prepare", [P, P, P, I, I, I, Z, Z, P, P, Z, P, ctypes.POINTER(I), P, Z, I, I, P])
    for dense in (True, False):                          # the next row's first columns behind a row's last, or a margin
        width = H if dense else H + 64
        x = torch.full((M + 1, width), 7.0, device="cuda")
        xg = torch.full((M + 1, width), 7.0, dtype=torch.bfloat16, device="cuda")
        ssq = torch.full(((H // 16 + 2) * K.SSQ_LD,), 7.0, device="cuda")
        x[:M, :H] = x0
        tiles = ctypes.c_int(0)                          # (rows in a wider room are for the C entry: the Python one takes dense rows)
        assert prepare(a.data_ptr(), w.data_ptr(), x.data_ptr(), M, H, 1024, 1024, width, gain.data_ptr(), xg.data_ptr(), width, ssq.data_ptr(),
                       ctypes.byref(tiles), None, 0, 0, 1, torch.cuda.current_stream().cuda_stream) == 0
        assert tiles.value == H // 16 and K.gemm_whole_pays(M, H, 1024, by16=True)
        assert off(x[:M, :H], x0.double() + y) < bound(1024)
        assert torch.equal(xg[:M, :H], (x[:M, :H] * gain).to(torch.bfloat16))
        squares = ssq.view(-1, K.SSQ_LD)[:H // 16, :M].double().sum(0)
        assert float((squares / (x[:M, :H].double() ** 2).sum(1) - 1).abs().max()) < bound(H)
        for t in (x[:, H:], x[M], xg[:, H:], xg[M], ssq[H // 16 * K.SSQ_LD:]):
            assert bool((t == 7.0).all())


# K of 7 and 13 chunks in runs of 3 and 4: the last run of a tile has a single chunk, and 1 / rms of a row is added up beside it
@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N,K_,runs", [(2048, 896, 3), (4096, 896, 3), (4096, 1664, 4)])
def test_a_prepared_norm_over_runs_of_one_chunk(M, N, K_, runs):
    from braidinfer_amd import kernels as K
    xg, _, w, y = operands(M, N, K_, M + N)
    tiles = K_ // 16
    ssq = torch.rand(tiles * K.SSQ_LD, device="cuda")
    scratch = torch.full((K.GEMM_SCRATCH_FLOATS,), float("nan"), device="cuda")
    assert K.gemm_wide_parts(M, N, K_, scratch.numel()) == runs
    want = y * torch.rsqrt(ssq.view(tiles, K.SSQ_LD)[:, :M].double().sum(0) / K_ + 1e-5)[:, None]
    out = torch.empty(M, N, device="cuda")
    K.gemm_norm_scaled(xg, ssq, tiles, 1e-5, w, out, scratch=scratch)
    assert off(out, want) < bound(K_) + 2 ** -24 * runs


@pytest.mark.parametrize("M,N,K_,pays", [(8, 6144, 4096, True), (8, 8192, 4096, True), (8, 8208, 4096, True), (16, 5120, 13824, True), (1, 28672, 4096, True), (24, 4096, 4096, True),
                                         (64, 4096, 4096, True), (64, 4096, 14336, False), (64, 28672, 4096, False), (67, 4096, 4096, True),
                                         (67, 4096, 14336, False), (67, 12288, 4096, False), (128, 2048, 2048, True), (129, 2048, 2048, False), (24, 4096, 4160, False),
                                         (65, 8192, 4096, True), (65, 8192, 14336, False), (72, 7168, 9216, False), (80, 2048, 4096, False), (96, 6144, 4096, True),
                                         (128, 8192, 5120, False), (65, 1024, 2048, True)])
def test_where_the_rule_takes_it(M, N, K_, pays):
    from braidinfer_amd import kernels as K
    assert K.gemm_whole_pays(M, N, K_) == pays
    a, _, w, want = operands(M, N, K_, 5)
    scratch = torch.full((K.GEMM_SCRATCH_FLOATS,), float("nan"), device="cuda")
    out, alone = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    K.gemm(a, w, out, scratch=scratch, whole=True)
    assert off(out, want) < bound(K_)
    if pays and M <= 16:                                 # a row's bits do not depend on the others
        K.gemm(a[:1], w, alone[:1], whole=True)
        assert torch.equal(alone[:1], out[:1])
    if pays and 16 < M <= 64:                            # unasked, the product's bits are those of the runs it may leave
        K.gemm(a, w, alone, scratch=scratch)
        runs = K.gemm_wide_partial(a, w, N, scratch)
        if runs:
            total = scratch[:M * N].clone()
            for r in range(1, runs):
                total += scratch[r * M * N:(r + 1) * M * N]
            assert torch.equal(total.view(M, N), alone)


# up to 16 rows, on both sides of the lines between tiles and resident workgroups: columns below and above one round, one chunk a wave and more
@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,K_,tiles", [(4096, 1024, False), (4100, 1024, True), (8192, 1024, True), (8194, 1024, False), (20480, 1024, False), (20480, 1152, True),
                                        (3072, 2048, True), (8208, 11008, True), (8208, 12288, False)])
def test_where_resident_workgroups_stay(M, N, K_, tiles):
    from braidinfer_amd import kernels as K
    assert K.gemm_whole_pays(M, N, K_) == tiles
    a, _, w, want = operands(M, N, K_, 7, blocked=N % 16 == 0 and N > 8192)
    out, one = torch.empty(M, N, device="cuda"), torch.empty(1, N, device="cuda")
    K.gemm(a, w, out)
    assert off(out, want) < bound(K_)
    half = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    K.gemm(a, w, half)
    assert torch.equal(half, out.to(torch.bfloat16))
    base = torch.randn(M, N, device="cuda")
    got, last = base.clone(), base[M - 1:].clone()
    K.gemm(a, w, got, accumulate=True)
    assert off(got, base.double() + want) < bound(K_)
    K.gemm(a[M - 1:], w, one)                            # a row's bits do not depend on the others
    K.gemm(a[M - 1:], w, last, accumulate=True)
    assert torch.equal(one, out[M - 1:]) and torch.equal(last, got[M - 1:])
    if N % 16 == 0:
        act = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
        K.gemm_swiglu(a, w, act)
        gu = want.view(M, N // 16, 2, 8)
        g, u = gu[:, :, 0].reshape(M, -1), gu[:, :, 1].reshape(M, -1)
        assert off(act, g / (1 + torch.exp(-g)) * u) < 2 ** -8


@pytest.mark.parametrize("M,N,K_", [(65, 4096, 4096), (128, 1028, 1024), (100, 2048, 2048)])
def test_one_run_left_for_the_norm(M, N, K_):
    from braidinfer_amd import kernels as K
    a, _, w, y = operands(M, N, K_, 9)
    x, gain = torch.randn(M, N, device="cuda"), torch.rand(N, device="cuda") + 0.5
    scratch = torch.full((K.GEMM_SCRATCH_FLOATS,), float("nan"), device="cuda")
    assert K.gemm_leave_runs(a, w, N, scratch) == 0 and K.gemm_leave_runs(a, w, N, scratch, True) == 1
    want = x.double() + y
    h = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    K.rmsnorm(x, gain, h, 1e-5, add=(scratch, 1))
    assert off(x, want) < bound(K_)
    assert off(h, want * torch.rsqrt((want ** 2).mean(1, keepdim=True) + 1e-5) * gain) < 2 ** -8
    assert K.gemm_leave_runs(a, w, N, scratch[:M * N - 4], True) == 0
