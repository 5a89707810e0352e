"""Which calls of ``linear.linear`` stay with the operator (no GPU needed)."""

from __future__ import annotations

import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode

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


@pytest.mark.parametrize("trace", ["make_fx", "jit", "flops"])
def test_traces_and_dispatch_modes_need_the_operator(trace):
    """Their operands may be plain tensors that hold real values."""
    x, w = _operands()
    seen = []

    def f(x, w):
        seen.append(linear._needs_operator(x, w))
        return torch.nn.functional.linear(x, w)

    if trace == "make_fx":
        make_fx(f, tracing_mode="real")(x, w)
    elif trace == "jit":
        torch.jit.trace(f, (x, w), check_trace=False)
    else:
        with FlopCounterMode(display=False):
            f(x, w)
    assert seen == [True]
    with torch.device("cpu"):  # a mode for new tensors only
        assert not linear._needs_operator(x, w)


@pytest.mark.parametrize("rows,N,K,taken", [
    (16, 2056, 512, True), (16, 24576, 4096, True), (17, 4096, 4096, False), (0, 4096, 4096, False),
    (1, 2048, 4096, False), (1, 4100, 4096, False), (1, 4096, 4097, False), (1, 4096, 256, False),
    (4, 4096, 8192, True), (5, 4096, 8192, False), (2, 4096, 12288, True), (3, 4096, 12288, False),
    (1, 4096, 12800, False), (2, 8200, 12288, True), (4, 12288, 4608, True),
    # over 4096 wide, more than one 16-column tile a CU and at most two
    (1, 4104, 4608, False), (4, 5120, 5120, False), (1, 6144, 8192, False), (2, 8192, 8192, False),
    (2, 8192, 12288, False), (16, 8192, 4096, True),
])
def test_sizes_given_to_the_kernel(rows, N, K, taken):
    assert linear._rows16_shape(rows, N, K) is taken
