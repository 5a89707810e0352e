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


def test_ranges_of_decode_and_prefill():
    """4 kv-heads of 4 heads on 256 CUs: the rule's branches and both of their bounds."""
    layer = mx.Attention(mx.AttentionArgs(64, 16, 4, 256, 64), device="cpu")
    layer._cus = 256
    ranges = {(1, 1, 128): 1, (1, 1, 192): 2, (1, 1, 1024): 8, (1, 1, 16384): 64, (4, 1, 4097): 13, (64, 1, 4096): 1,
              (1, 4, 300): 3, (1, 8, 127): 1, (1, 8, 16384): 64, (1, 64, 8256): 26, (32, 8, 4096): 4,
              (1, 128, 128): 1, (1, 128, 8320): 15, (1, 512, 4608): 4, (1, 4096, 4096): 1}
    assert {k: layer._splits(*k) for k in ranges} == ranges
