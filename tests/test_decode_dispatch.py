"""Which decode steps ``gdn_conv_decode`` takes (no GPU needed: it leaves a
call to the two launches before it looks for a device)."""

from __future__ import annotations

import pytest
import torch

from multiplex_amd import conv

D = 128


@pytest.mark.parametrize("B,Hk,Hv,taken", [
    (1, 16, 32, True), (64, 16, 32, True), (65, 2, 4, False), (64, 2, 4, True),
    (32, 16, 64, True), (33, 16, 64, False), (64, 16, 64, False), (16, 16, 128, True), (17, 16, 128, False),
])
def test_rows_and_heads(B, Hk, Hv, taken):
    C = (2 * Hk + Hv) * D
    bf = dict(dtype=torch.bfloat16)
    gates = torch.zeros(B, 1, Hv, **bf)
    args = (torch.zeros(B, 1, C, **bf), torch.zeros(C, 4, **bf), Hk, Hv, D, D, gates, gates, torch.zeros(Hv),
            torch.zeros(Hv), None, None)
    if taken:
        with pytest.raises(ValueError):  # the operands are not on a device
            conv.gdn_conv_decode(*args)
    else:
        assert conv.gdn_conv_decode(*args) is None
