"""Which calls of ``linear.linear`` stay with the operator (no GPU needed)."""

from __future__ import annotations

import pytest
import torch
import torch.autograd.forward_ad as fwad

from multiplex_amd import linear


def _operands():
    return torch.randn(4, 8), torch.randn(6, 8)


def test_plain_operands_do_not_need_the_operator():
    x, w = _operands()
    assert not linear._needs_operator(x, w)
    p = torch.nn.Parameter(w)
    assert linear._needs_operator(x, p)
    with torch.no_grad():
        assert not linear._needs_operator(x, p)
        with fwad.dual_level():
            assert not linear._needs_operator(x, w)


@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_tangents_need_the_operator(grad):
    x, w = _operands()
    with torch.set_grad_enabled(grad), fwad.dual_level():
        assert linear._needs_operator(fwad.make_dual(x, torch.ones_like(x)), w)
        assert linear._needs_operator(x, fwad.make_dual(w, torch.ones_like(w)))


@pytest.mark.parametrize("transform", ["jvp", "vjp", "vmap"])
def test_function_transforms_need_the_operator(transform):
    x, w = _operands()
    seen = []

    def f(w):
        seen.append(linear._needs_operator(x, w))
        return torch.nn.functional.linear(x, w)

    if transform == "jvp":
        torch.func.jvp(f, (w,), (w,))
    elif transform == "vjp":
        torch.func.vjp(f, w)
    else:
        torch.func.vmap(f)(w[None])
    assert seen == [True]
