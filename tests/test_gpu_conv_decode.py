"""``gdn_conv_decode`` (the conv prologue and one recurrent step in one launch)
against the two launches it stands for: the same arithmetic in the same
order, so y, the states and the conv states are equal bit for bit."""

from __future__ import annotations

import math

import pytest
import torch

import multiplex_amd as mx
from multiplex_amd import conv

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def _inputs(B, Hk, Hv, params=torch.float32, cs=True, state=True):
    gen = torch.Generator().manual_seed(B + 10 * Hk + Hv)
    C = 2 * Hk * D + Hv * D
    wide = torch.randn(B, 1, C + 8 + 8 * Hv, generator=gen).to(torch.bfloat16).to(DEV)
    t = dict(qkv=wide[..., :C], a=wide[..., C + 8:C + 8 + Hv], b=wide[..., C + 8 + Hv:C + 8 + 2 * Hv],
             w=(torch.randn(C, 4, generator=gen) * 0.3).to(torch.bfloat16).to(DEV),
             A_log=(torch.rand(Hv, generator=gen) * math.log(16.0)).to(params).to(DEV),
             dt_bias=(torch.rand(Hv, generator=gen) * 2 - 1).to(params).to(DEV),
             cs=torch.randn(B, 3, C, generator=gen).to(torch.bfloat16).to(DEV) if cs else None,
             state=(torch.randn(B, Hv, D, D, generator=gen) * 0.1).to(DEV) if state else None)
    return t


def _step(t, Hk, Hv, **kw):
    return conv.gdn_conv_decode(t["qkv"], t["w"], Hk, Hv, D, D, t["a"], t["b"], t["A_log"], t["dt_bias"], t["state"],
                                t["cs"], **kw)


# batches and heads on both sides of the lines between 2, 4 and 8 units a wave, groups of 1 to 4
@pytest.mark.parametrize("B,Hk,Hv,params,cs,state", [
    (1, 16, 32, torch.float32, True, True),
    (4, 16, 32, torch.bfloat16, True, True),
    (7, 16, 32, torch.float32, False, True),
    (8, 16, 32, torch.float32, True, False),
    (64, 4, 4, torch.bfloat16, False, False),
    (5, 1, 3, torch.float32, True, True),
    (64, 4, 16, torch.float32, True, True),
])
def test_equals_prologue_and_step(B, Hk, Hv, params, cs, state):
    t = _inputs(B, Hk, Hv, params, cs, state)
    y, s, c = _step(t, Hk, Hv)
    q, k, v, c2 = mx.gdn_conv_prologue(t["qkv"], t["w"], Hk, Hv, D, D, t["cs"])
    y2, s2 = mx.gated_delta_update(q, k, v, t["a"], t["b"], t["A_log"], t["dt_bias"], t["state"])
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(s, s2) and torch.equal(c, c2)
    y, s, c = _step(t, Hk, Hv, write_conv_state=False)
    assert c is None and torch.equal(y, y2) and torch.equal(s, s2)


def test_leaves_other_operands_to_the_two_launches():
    t = _inputs(3, 2, 4)
    assert _step(t, 2, 4) is not None
    for change in (dict(w=t["w"].float()), dict(qkv=t["qkv"].half()), dict(state=t["state"][..., :64]),
                   dict(cs=t["cs"][:, :2]), dict(dt_bias=t["dt_bias"].to(torch.bfloat16)),
                   dict(b=t["b"].contiguous()), dict(state=t["state"].transpose(2, 3)),
                   dict(A_log=t["A_log"].half(), dt_bias=t["dt_bias"].half())):
        assert _step(dict(t, **change), 2, 4) is None
    assert _step(_inputs(65, 2, 4), 2, 4) is None
