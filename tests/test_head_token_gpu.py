"""Single tokens of the gated recurrences, normed by heads in one launch, against the walk and the head norm."""
import pytest
import torch

from braidinfer_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d,e", [(3, 64, 64), (1, 4, 4), (5, 20, 12), (2, 60, 68), (3, 68, 64), (2, 128, 128), (2, 124, 100)])
def test_single_tokens_in_one_launch(H, d, e, dtype):
    """Heads at and beside the widths a wave's blocks and a lane's rows hold; a padding sequence among the others; the
    state's slots in no order, with floats behind the heads' that stay as they are.  The sums have the order of the
    two launches', so results are the same bits."""
    g = torch.Generator().manual_seed(H * d + e)
    B, slots = 5, [3, -1, 0, 4, 2]
    rows = torch.randn(B, 3 * H * d + 2 * H * e + 4, generator=g).cuda()
    gate = rows[:, 3 * H * d + H * e:3 * H * d + 2 * H * e]
    w0, u = torch.randn(H * d, generator=g).cuda(), torch.randn(H * d, generator=g).cuda()
    norm_w = torch.randn(H * e, generator=g).cuda()
    n = 1
    for k in K.glr_state_shape(H, d, e):
        n *= k
    first = torch.randn(6, n + 7, generator=g).cuda()
    states = [first.clone(), first.clone()]
    ys = [torch.full((B, H * e), 5.0, device="cuda", dtype=dtype) for _ in range(2)]
    at = torch.tensor(slots, dtype=torch.int32, device="cuda")
    cu = torch.arange(B + 1, dtype=torch.int32, device="cuda")
    assert K.head_token_takes(d, e)
    for _ in range(2):                             # the second token from the state that the first left
        o = torch.full((B, H * e), 7.0, device="cuda")
        K.wkv_scan(rows, w0, u, o, states[0], cu, at, B, H, d, e)
        K.head_norm_gate(o, norm_w, gate, ys[0], H, e, 1e-5)
        K.wkv_scan(rows, w0, u, o, states[1], cu, at, B, H, d, e, normed=(norm_w, gate, ys[1], 1e-5))
        assert torch.equal(ys[0], ys[1]) and torch.equal(states[0], states[1])
    assert (ys[1][1] == 0).all() and not torch.equal(states[1], first)


@pytest.mark.parametrize("biased", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d,e", [(3, 64, 64), (1, 4, 4), (5, 20, 12), (2, 60, 68), (3, 68, 64), (2, 128, 128), (2, 124, 100)])
def test_single_tokens_without_a_bonus(H, d, e, dtype, biased):
    """The same of the recurrence whose gates may have biases and bounds, and its norm a weight, or none of them."""
    g = torch.Generator().manual_seed(H * d + e + 1)
    B, slots = 5, [3, -1, 0, 4, 2]
    live = torch.tensor([b for b in range(B) if slots[b] >= 0], device="cuda")
    rows = torch.randn(B, 2 * H * d + H * e, generator=g).cuda()
    f_bias, lower = (torch.randn(H * d, generator=g).cuda(), torch.rand(H * d, generator=g).cuda()) if biased else (None, None)
    norm_w = torch.randn(e, generator=g).cuda() if biased else None
    first = torch.randn((6,) + tuple(K.glr_state_shape(H, d, e)), generator=g).cuda()
    states = [first.clone(), first.clone()]
    ys = [torch.full((B, H * e), 5.0, device="cuda", dtype=dtype) for _ in range(2)]
    at = torch.tensor(slots, dtype=torch.int32, device="cuda")
    cu = torch.arange(B + 1, dtype=torch.int32, device="cuda")
    for _ in range(2):
        o = torch.zeros((B, H * e), device="cuda")
        K.glr_scan(rows, f_bias, lower, o, states[0], cu, at, B, H, d, e)
        K.head_rmsnorm(o, norm_w, ys[0], H, e, 1e-5)
        K.glr_scan(rows, f_bias, lower, o, states[1], cu, at, B, H, d, e, normed=(norm_w, ys[1], 1e-5))
        assert torch.equal(ys[0][live], ys[1][live]) and torch.equal(states[0], states[1])
    assert (ys[1][1] == 0).all() and not torch.equal(states[1], first)


@pytest.mark.parametrize("d,e", [(130, 64), (64, 132), (6, 8), (8, 6), (0, 8)])
def test_other_widths_are_refused(d, e):
    assert not K.head_token_takes(d, e)


def test_vectors_at_odd_places_are_refused():
    """A checkpoint's vectors may be views that start anywhere."""
    v = torch.zeros(132, device="cuda")
    assert K.head_token_takes(64, 64, v, None, v[4:68]) and not K.head_token_takes(64, 64, v, v[1:65])
