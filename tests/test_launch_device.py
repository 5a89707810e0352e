"""Launches go to the device of their tensors, whichever is current.

A device's default stream is handle 0, and a launch on handle 0 runs on the
current device, so every launch enters its tensors' device.  Checked without a
GPU: the library call and the device context are replaced by stand-ins.
"""

from __future__ import annotations

import contextlib

import pytest
import torch

import multiplex_amd as mx
from multiplex_amd import _lib, attention, gated_delta, linear


@pytest.fixture
def launches(monkeypatch):
    """The names of the library calls made, each inside its device's context."""
    inside, made = [], []

    @contextlib.contextmanager
    def enter(dev):
        inside.append(dev)
        yield
        inside.pop()

    def call(name, *args):
        assert inside, f"{name} is launched on whichever device is current"
        made.append(name)

    monkeypatch.setattr(_lib, "call", call)
    for mod in (attention, linear):
        monkeypatch.setattr(mod, "_on_device", enter, raising=False)
        monkeypatch.setattr(mod, "_stream", lambda dev: 0)
        monkeypatch.setattr(mod, "_require_device", lambda tensors, names: torch.device("cpu"))
    return made


def test_on_device_enters_another_device_only(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert isinstance(gated_delta._on_device(torch.device("cuda", 0)), contextlib.nullcontext)
    other = gated_delta._on_device(torch.device("cuda", 1))
    assert isinstance(other, torch.cuda.device) and other.idx == 1


class _Offsets:
    """A KV cache's offsets on a device."""

    is_cuda, dtype, device = True, torch.int32, torch.device("cuda", 1)

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 0

    def numel(self):
        return 3


def test_cache_offsets(launches):
    c = mx.KVCache(3, 1, 128, 256, "cpu")
    c.pos0 = _Offsets()
    c.advance(5)
    c.trim(2)
    assert c.lengths == [3, 3, 3] and launches == ["gdn_pos_add"] * 2


def test_projection_of_few_rows(launches):
    x, w = torch.zeros(3, 1, 512, dtype=torch.bfloat16), torch.zeros(2056, 512, dtype=torch.bfloat16)
    assert linear._rows16(x, w, 3).shape == (3, 1, 2056)
    assert launches == ["gdn_linear_rows16"]
