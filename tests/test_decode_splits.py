"""Into how many runs single-token attention cuts a sequence's pages: the rule alone."""
import pytest

from braidinfer_amd.parts.attention import decode_splits


@pytest.mark.parametrize("batch,bound,runs", [(17, 768, 1), (17, 1024, 2), (17, 1900, 2), (20, 1024, 1), (20, 1408, 2), (24, 1024, 1), (24, 1900, 2),
                                              (31, 1900, 1), (31, 3072, 2), (32, 2048, 1), (32, 3072, 2), (33, 4096, 1), (64, 4096, 1),
                                              (16, 1408, 2), (16, 1900, 4), (9, 1900, 4), (8, 1024, 4), (8, 2048, 8), (5, 1024, 4), (3, 2048, 8),
                                              (1, 64, 1), (1, 128, 1), (2, 256, 2), (40, 64 * 65, 2)])
def test_runs_by_sequences_and_bound(batch, bound, runs):
    """8 kv heads, 256 compute units: one run or two by the share of units that one would take; the same for the heads of
    half as many kv heads of twice the sequences."""
    assert decode_splits(batch, 8, bound, 64) == decode_splits(2 * batch, 4, bound, 64) == runs
