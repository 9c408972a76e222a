"""Which rows an RMS norm takes into the kernel that adds a product's runs: the rule alone, on the host."""
import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.engine.step import Workspace
from braidinfer_amd.parts.base import Norm, NormedInput, ResidualSink
from braidinfer_amd.parts.linear import linear
from braidinfer_amd.parts.norm import RMSNorm


@pytest.mark.parametrize("rows,x_off,w_off,taken", [(64, 0, 0, None), (65, 0, 0, True), (1024, 0, 0, True), (1025, 0, 0, None), (100, 1, 0, False),
                                                    (100, 0, 2, False), (100, 4, 8, True)])
def test_rows_and_weights_off_16_bytes_keep_their_two_kernels(monkeypatch, rows, x_off, w_off, taken):
    """taken: the runs are left and normed in one pass; False: nothing is launched, and the product and the norm run by themselves."""
    called = []
    monkeypatch.setattr(K, "gemm_leave_runs", lambda *a: called.append("runs") or 3)
    monkeypatch.setattr(K, "gemm_stream_takes", lambda *a: False)
    monkeypatch.setattr(K, "rmsnorm", lambda x, w, out, eps, rows=None, add=None: called.append("norm" if add is None else "sum and norm"))
    n, k = 256, 128
    norm = RMSNorm(n, 1e-5)
    norm.weight = torch.ones(n + w_off)[w_off:]
    x = torch.zeros(rows * n + x_off)[x_off:].view(rows, n)
    a, w = torch.zeros(rows, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.bfloat16)
    prepared = norm.prepare_in_product(a, w, x, Workspace("cpu"))
    if taken:
        assert called == ["runs", "sum and norm"] and norm.rows_of_prepared(prepared).shape == (rows, n)
    else:
        assert called == [] and prepared is None


@pytest.mark.parametrize("whole", [True, False])
def test_a_norm_with_a_product_of_its_own(whole):
    """A norm from outside gives what it prepared and takes (prepared, w, out) back, whichever bits the product is asked for."""
    class Own(Norm):
        def prepare_in_product(self, a, w, x, ws):
            return "mine"

        def product_of_prepared(self, prepared, w, out, swiglu=False):
            assert prepared == "mine" and not swiglu
            out.fill_(3.0)
            return True
    norm, x, w, out = Own(), torch.zeros(4, 8), torch.zeros(6, 8), torch.zeros(4, 6)
    sink = ResidualSink(x, norm)
    linear(torch.zeros(4, 8), torch.zeros(8, 8), sink, Workspace("cpu"), accumulate=True)
    linear(NormedInput(x, norm, Workspace("cpu"), torch.float32, sink.prepared), w, out, Workspace("cpu"), whole=whole)
    assert (out == 3.0).all()
