"""The rules by which a step chooses its launches: the spans an attention launch walks, the fused sequence over FP8."""

from __future__ import annotations

import pytest

from btb_amd.decode import fp8_step_fused, pass_spans, step_on_spans, step_spans


@pytest.mark.parametrize("T", [2, 3, 16, 17, 32])
@pytest.mark.parametrize("Hq,Hk", [(1, 1), (8, 1), (4, 2), (16, 2), (32, 4), (32, 8), (64, 8), (8, 8), (512, 256)])
@pytest.mark.parametrize("cap", [1, 127, 128, 129, 4608, 35200, 131072, 2000000])
def test_a_passs_spans_cover_the_cache_in_whole_batches(T, Hq, Hk, cap):
    S = pass_spans(256, T, Hq, Hk, cap)
    span = -(-(-(-cap // S)) // 128) * 128  # as the library rounds it
    assert 1 <= S * (Hq // Hk) <= 1024
    assert S * span >= cap and (S - 1) * span < cap


@pytest.mark.parametrize("T", [2, 4, 17, 32])
@pytest.mark.parametrize("Hq,Hk", [(1, 1), (8, 1), (4, 2), (16, 2), (9, 3), (32, 4)])
@pytest.mark.parametrize("cap", [8192, 8193, 16384, 33024, 70016, 2000000])
def test_a_passs_spans_stay_with_the_fast_fold(T, Hq, Hk, cap):
    """(an odd number of states is left to the kernels that cut as many spans as the fold takes)"""
    assert pass_spans(256, T, Hq, Hk, cap) <= 64 or T * Hq % 2 == 1


@pytest.mark.parametrize("Hq,Hk", [(1, 1), (8, 1), (4, 2), (16, 2), (32, 4), (32, 8), (8, 8), (512, 256), (12, 4)])
@pytest.mark.parametrize("cap", [64, 8191, 8192, 16383, 16384, 35200, 1000000])
def test_a_steps_spans_cover_the_cache(Hq, Hk, cap):
    S = step_on_spans(256, Hq, Hk, cap)
    if Hq // Hk == 3 or cap < 8192:
        assert S == 0
    if S:
        span = -(-(-(-cap // S)) // 128) * 128
        assert S <= 64 and S * Hq % 2 == 0 and S * span >= cap and (S - 1) * span < cap


@pytest.mark.parametrize("Hq,Hk", [(8, 8), (16, 8), (32, 8), (64, 8), (16, 4), (32, 4), (8, 2), (16, 2), (4, 2), (8, 4)])
@pytest.mark.parametrize("cap", [8192, 8800, 12288, 16384, 20000, 35200, 131072])
def test_a_step_walks_its_spans_where_they_are_short_for_it(Hq, Hk, cap):
    """the walk's batch of keys costs up to one and a half of the register kernel's, whose own batches have to be many - or
    its spans, which are slow to fold beyond 64"""
    S, others = step_on_spans(256, Hq, Hk, cap), step_spans(256, Hq, Hk, cap)
    ours, theirs = -(-cap // (min(64, 256 // Hk) * 128)), -(-cap // (others * 128))
    pays = Hq // Hk >= 4 and theirs >= 3 and 3 * ours <= 2 * theirs
    assert bool(S) == (others > 64 or pays)
    if S:
        assert -(-(-(-cap // S)) // 128) == ours


@pytest.mark.parametrize("T,hidden,fused", [(1, 4096, True), (2, 3072, True), (2, 3073, False), (2, 4096, False), (2, 4224, True),
                                            (3, 1024, False), (1, 40960, True), (1, 40961, False), (2, 27306, True),
                                            (2, 27392, False)])
def test_fp8_steps_that_fit_and_pay(T, hidden, fused):
    assert fp8_step_fused(T, hidden) == fused
