"""The rules that cut a cache into the spans an attention launch walks."""

from __future__ import annotations

import pytest

from btb_amd.decode import pass_spans, step_on_spans


@pytest.mark.parametrize("T", [2, 3, 16, 17, 32])
@pytest.mark.parametrize("Hq,Hk", [(1, 1), (8, 1), (4, 2), (16, 2), (32, 4), (32, 8), (64, 8), (8, 8), (512, 256)])
@pytest.mark.parametrize("cap", [1, 127, 128, 129, 4608, 35200, 131072, 2000000])
def test_a_passs_spans_cover_the_cache_in_whole_batches(T, Hq, Hk, cap):
    S = pass_spans(256, T, Hq, Hk, cap)
    span = -(-(-(-cap // S)) // 128) * 128  # as the library rounds it
    assert 1 <= S * (Hq // Hk) <= 1024
    assert S * span >= cap and (S - 1) * span < cap


@pytest.mark.parametrize("Hq,Hk", [(1, 1), (8, 1), (4, 2), (16, 2), (32, 4), (32, 8), (8, 8), (512, 256), (12, 4)])
@pytest.mark.parametrize("cap", [64, 8191, 8192, 16383, 16384, 35200, 1000000])
def test_a_steps_spans_cover_the_cache(Hq, Hk, cap):
    S = step_on_spans(256, Hq, Hk, cap)
    if Hq // Hk == 3 or cap < 8192:
        assert S == 0
    if S:
        span = -(-(-(-cap // S)) // 128) * 128
        assert S <= 64 and S * Hq % 2 == 0 and S * span >= cap and (S - 1) * span < cap
