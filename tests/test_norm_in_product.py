"""Which rows an RMS norm takes into the kernel that adds a product's runs: the rule alone, on the host."""
import pytest
import torch

from braidinfer_amd import kernels as K
from braidinfer_amd.engine.step import Workspace
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
