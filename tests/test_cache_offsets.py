"""A KV cache's offsets without memory of their own (no GPU needed)."""

from __future__ import annotations

from torch._subclasses.fake_tensor import FakeTensorMode

import multiplex_amd as mx


def test_offsets_of_a_fake_cache_advance_and_roll_back():
    """Shapes and sizes of a cache may be worked out under a fake mode, whose device tensors hold no memory."""
    with FakeTensorMode():
        c = mx.KVCache(2, 1, 128, 256, "cuda")
        c.advance(7)
        assert c.pos0.is_cuda and c.trim(3) == 3
        assert c.lengths == [4, 4] and c.pos0.shape == (2,)
