"""The recurrences' form for steps of single tokens: tokens fed one a step leave the same bits, in outputs and states, as the walk
over all of them at once, at head sizes around the lanes' rows and the 16-byte loads."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(gen, *shape):
    return torch.randn(*shape, generator=gen).cuda()


def _one_by_one(walk, shape, T, B):
    """walk(rows of the step, cu, slots, state) -> outputs: all tokens of the first B sequences at once, and one a step, a
    padding sequence among them."""
    g = torch.Generator().manual_seed(T)
    first = _rand(g, B + 2, *shape)
    slots = torch.tensor([B, 0, -1][:B] + [-1], dtype=torch.int32).cuda()            # B 2: slots 2, 0 and padding
    rows = torch.arange((B + 1) * T).reshape(B + 1, T)
    whole, single = first.clone(), first.clone()
    cu = (torch.arange(B + 2) * T).int().cuda()
    outs = walk(rows.reshape(-1).cuda(), cu, slots, whole)
    for t in range(T):
        got = walk(rows[:, t].contiguous().cuda(), torch.arange(B + 2).int().cuda(), slots, single)
        for a, b in zip(outs, got):
            assert torch.equal(a.reshape(B + 1, T, -1)[:B, t], b.reshape(B + 1, -1)[:B])
    assert torch.equal(whole, single) and not torch.equal(whole, first)
    assert torch.equal(whole[1], first[1])                                           # a slot that nobody named


@pytest.mark.parametrize("mode", ["delta", "channels", "weighted", "weighted with sum", "fixed", "fixed silu"])
@pytest.mark.parametrize("H,G,d,e", [(2, 1, 128, 128), (3, 3, 16, 20), (2, 2, 65, 33), (1, 1, 130, 5), (1, 1, 257, 16), (2, 1, 60, 3)])
def test_outer_sums(mode, H, G, d, e):
    from braidinfer_amd import kernels as K
    T, B, g = 5, 2, torch.Generator().manual_seed(d)
    n, extra = (B + 1) * T, mode == "weighted with sum"
    if mode.startswith("fixed"):
        G = H
    q, k = _rand(g, n, G * d) / d ** 0.5, _rand(g, n, G * d) / d ** 0.5
    v, gb, gc, dec = _rand(g, n, H * e), torch.rand(n, 2 * H, generator=g).cuda(), torch.rand(n, H * d, generator=g).cuda(), torch.rand(H, generator=g).cuda()
    skip = _rand(g, H)

    def walk(rows, cu, slots, state):
        at = lambda x: x[rows].contiguous()
        out = torch.zeros(len(rows), H * e, device="cuda")
        n_out = torch.zeros(len(rows), H, device="cuda") if extra else None
        fixed = mode.startswith("fixed")
        K.dr_scan(at(q), at(k), at(v), None if fixed else at(gb), dec if fixed else None, out, state, cu, slots, B + 1, H, G, d, e,
                  silu=mode == "fixed silu", gc=at(gc) if mode == "channels" else None, weighted=mode.startswith("weighted"),
                  skip=skip if mode == "weighted" else None, n_out=n_out)
        return [out] + ([n_out] if extra else [])
    _one_by_one(walk, K.glr_state_shape(H, d, e + extra), T, B)


@pytest.mark.parametrize("gates", [False, True])
@pytest.mark.parametrize("H,d,e", [(2, 128, 128), (3, 16, 20), (2, 65, 33), (1, 130, 5), (1, 257, 16), (2, 60, 3)])
def test_gated(gates, H, d, e):
    from braidinfer_amd import kernels as K
    T, B, g = 5, 2, torch.Generator().manual_seed(d)
    rows_all = _rand(g, (B + 1) * T, 2 * H * d + H * e)
    bias, lower = (_rand(g, H * d), torch.rand(H * d, generator=g).cuda()) if gates else (None, None)

    def walk(rows, cu, slots, state):
        out = torch.zeros(len(rows), H * e, device="cuda")
        K.glr_scan(rows_all[rows].contiguous(), bias, lower, out, state, cu, slots, B + 1, H, d, e)
        return [out]
    _one_by_one(walk, K.glr_state_shape(H, d, e), T, B)


def test_gates_at_any_address():
    """Biases and bounds at odd multiples of 4 bytes (the chunks' walk takes those): the same bits as at multiples of 16."""
    from braidinfer_amd import kernels as K
    H, d, e, B = 3, 64, 32, 5
    g = torch.Generator().manual_seed(1)
    rows, first = _rand(g, B, 2 * H * d + H * e), _rand(g, B, *K.glr_state_shape(H, d, e))
    vectors = [_rand(g, H * d + 4), torch.rand(H * d + 4, generator=g).cuda()]
    cu, slots = torch.arange(B + 1, dtype=torch.int32).cuda(), torch.arange(B, dtype=torch.int32).cuda()

    def run(bias, lower):
        out, state = torch.zeros(B, H * e, device="cuda"), first.clone()
        K.glr_scan(rows, bias, lower, out, state, cu, slots, B, H, d, e)
        return out, state
    moved = [v[1:1 + H * d] for v in vectors]
    dense = [v.clone() for v in moved]
    want = run(*dense)
    for got in (run(*moved), run(moved[0], dense[1]), run(dense[0], moved[1])):
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
