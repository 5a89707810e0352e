"""The key ranges an attention layer asks for (no GPU needed)."""

from __future__ import annotations

import pytest
import torch

import multiplex_amd as mx


@pytest.mark.parametrize("Hq,Hkv,D", [(16, 4, 256), (8, 2, 256), (16, 16, 128), (24, 1, 128)])
def test_every_range_holds_keys_and_lies_on_whole_blocks(Hq, Hkv, D):
    layer = mx.Attention(mx.AttentionArgs(64, Hq, Hkv, D, 64), device="cpu")
    layer._cus = 256
    for B in (1, 2, 4, 7, 64, 300):
        for T in (1, 2, 5, 16, 63, 64, 130, 512, 1000):
            for past in (0, 1, 63, 64, 127, 128, 129, 500, 1023, 2047, 4000, 4096, 16383):
                L = past + T
                n = layer._splits(B, T, L)
                keys = -(-(-(-L // n)) // 64) * 64  # a range's length in gdn_attn_fwd
                assert n >= 1 and (n - 1) * keys < L, (B, T, L, n)
    assert layer._splits(1, 0, 0) == 1


@pytest.mark.parametrize("T", [1, 8, 200])
def test_a_batch_of_no_rows_takes_one_range(T):
    """(All of its requests have left.)"""
    assert _ranges(16, 4, 256, [(0, T, T), (0, T, 5000)]) == {(0, T, T): 1, (0, T, 5000): 1}


def _ranges(Hq, Hkv, D, calls):
    layer = mx.Attention(mx.AttentionArgs(64, Hq, Hkv, D, 64), device="cpu")
    layer._cus = 256
    return {k: layer._splits(*k) for k in calls}


def test_ranges_of_decode_and_prefill():
    """4 kv-heads of 4 heads on 256 CUs, (B, T, keys): the rule's branches and both of their bounds."""
    ranges = {(1, 1, 128): 1, (1, 1, 256): 2, (1, 1, 1024): 8, (1, 1, 16384): 64, (4, 1, 4097): 13, (64, 1, 4096): 1,
              (1, 4, 300): 3, (1, 8, 127): 1, (1, 8, 16384): 64, (1, 64, 8256): 26, (32, 8, 4096): 4,
              (1, 128, 128): 1, (1, 128, 8320): 15, (1, 512, 4608): 4, (1, 4096, 4096): 1}
    assert _ranges(16, 4, 256, ranges) == ranges


def test_ranges_whose_partial_results_do_not_pay():
    """One range each: two of them took 1.13 to 1.59 times as long."""
    for heads, calls in {(16, 4, 128): [(1, 1, 196), (16, 1, 256), (4, 100, 295), (16, 64, 576), (4, 256, 768),
                                        (4, 256, 1256), (1, 1024, 1536)],
                         (8, 2, 256): [(16, 64, 259), (16, 128, 640)], (16, 4, 256): [(16, 32, 287)]}.items():
        assert set(_ranges(*heads, calls).values()) == {1}


def test_more_workgroups_than_compute_units_take_long_ranges():
    """(B, T, keys) of 56 and 96 workgroups a range: the fifth (third) range would leave the others' CUs idle
    (41 us against 33, 17.8 against 15.3 for one)."""
    assert _ranges(32, 8, 256, [(7, 1, 2501), (7, 1, 4096)]) == {(7, 1, 2501): 4, (7, 1, 4096): 5}
    assert _ranges(8, 2, 256, [(48, 1, 385)]) == {(48, 1, 385): 2}
