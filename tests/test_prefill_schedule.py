"""The host rule that cuts a prefill launch into key ranges (CPU)."""
import pytest

from muserve_amd import _lib
from muserve_amd.kernels.attention import prefill_schedule

CUS = 256


@pytest.mark.parametrize("batch,max_q,max_k", [
    (8, 1, 13916), (8, 20, 13932), (2, 1, 51120), (2, 64, 51183), (32, 40, 3900)])
def test_short_chunks_on_long_prefixes_take_the_grid(batch, max_q, max_k):
    """One query tile per sequence and ranges of at most 8 key tiles: a plan
    costs a launch and saves nothing."""
    splits, split_len, planned = prefill_schedule(batch * max_q, max_q, max_k, batch, 1, True, CUS)
    assert not planned
    assert 64 * 4 <= split_len <= 64 * 8 and splits * split_len >= max_k


@pytest.mark.parametrize("max_q,max_k", [(1, 59467), (64, 59517), (64, 120000), (200, 16018)])
def test_ranges_of_one_row_are_bounded(max_q, max_k):
    """The merge walks a row's ranges serially: past 64 they get longer."""
    splits, split_len, planned = prefill_schedule(max_q, max_q, max_k, 1, 1, True, CUS)
    assert not planned and splits * split_len >= max_k
    assert splits <= 64 or split_len >= 64 * 8


@pytest.mark.parametrize("batch,n,one", [(8, 300, True), (8, 500, True), (4, 300, True),
                                         (4, 700, False), (1, 300, False), (1, 2000, False)])
def test_ranges_without_a_mask_pay_for_their_merge(batch, n, one):
    splits, _, planned = prefill_schedule(batch * n, n, n, batch, 1, False, CUS)
    assert not planned and (splits == 1) == one


def test_every_schedule_is_one_the_library_takes():
    """Over the range of sizes: workspace sizes exist, ranges cover the keys."""
    lib = _lib.load()
    n = 0
    for heads in (1, 2, 4):
        for batch in (1, 2, 3, 7, 8, 9, 31, 64, 255, 300, 1100):
            for max_q in (1, 16, 33, 64, 65, 200, 1000, 4096):
                for prefix in (0, 1, 63, 500, 3000, 16384, 60000, 1 << 20):
                    for causal in (True, False):
                        tokens = max(max_q, batch * max_q // 2)
                        max_k = max_q + prefix
                        splits, split_len, planned = prefill_schedule(
                            tokens, max_q, max_k, batch, heads, causal, CUS)
                        assert splits >= 1 and splits * heads <= 65535
                        if planned:
                            assert lib.mkv_prefill_attention_plan_bytes(
                                tokens, 4 * heads, heads, batch, max_q, splits) > 0
                        elif splits > 1:
                            assert split_len % 64 == 0 and splits * split_len >= max_k
                            assert lib.mkv_prefill_attention_workspace_bytes(
                                tokens, 4 * heads, splits) > 0
                        n += 1
    assert n == 3 * 11 * 8 * 8 * 2
