"""Launches go to the device of their tensors, whichever is current.

A device's default stream is handle 0, and a launch on handle 0 runs on the
current device, so every launch enters its tensors' device.  Checked without a
GPU: the library call and the device context are replaced by stand-ins.
"""

from __future__ import annotations

import contextlib

import pytest
import torch

from multiplex_amd import _lib, attention, conv, epilogue, gated_delta, linear


class _Library:
    """The library, with every launch given to ``call`` by its name."""

    def __init__(self, call):
        self._call = call

    def __getattr__(self, name):
        if name.endswith("_workspace_bytes"):
            return lambda *sizes: 64
        return lambda *args: self._call(name)


@pytest.fixture
def launches(monkeypatch):
    """The names of the launches made, each with its tensors' device current, which device 0 is before."""
    inside, made = [], []

    @contextlib.contextmanager
    def enter(dev):
        inside.append(dev)
        yield
        inside.pop()

    def call(name):
        assert inside, f"{name} is launched on whichever device is current"
        made.append(name)
        return _lib.OK

    monkeypatch.setattr(_lib, "_current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "device", enter)
    monkeypatch.setattr(_lib, "_lib", _Library(call))
    monkeypatch.setattr(_lib, "_recurrent", lambda packed: call("gdn_recurrent"))
    for mod in (attention, conv, epilogue, gated_delta, linear):
        monkeypatch.setattr(mod, "_stream", lambda dev: 0)
        monkeypatch.setattr(mod, "_require_device", lambda tensors, names: torch.device("cpu"))
    return made


def test_on_device_enters_another_device_only(monkeypatch):
    monkeypatch.setattr(_lib, "_current_device", lambda: 0)
    assert isinstance(_lib.on_device(torch.device("cuda", 0)), contextlib.nullcontext)
    other = _lib.on_device(torch.device("cuda", 1))
    assert isinstance(other, torch.cuda.device) and other.idx == 1


def test_cache_offsets(launches):
    attention._pos_add(torch.zeros(3, dtype=torch.int32), 5, 0)
    assert launches == ["gdn_pos_add"]


def test_projection_of_few_rows(launches):
    x, w = torch.zeros(3, 1, 512, dtype=torch.bfloat16), torch.zeros(2056, 512, dtype=torch.bfloat16)
    assert linear._rows16(x, x.data_ptr(), w.data_ptr(), 3, 2056, 512).shape == (3, 1, 2056)
    assert launches == ["gdn_linear_rows16"]


def _bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


def test_attention_launches(launches):
    cache = _bf16(2, 1, 64, 128)
    pos0 = torch.zeros(2, dtype=torch.int32)
    q = attention.attn_qk(_bf16(2, 1, 512), _bf16(2, 1, 128), _bf16(2, 1, 128), _bf16(128), _bf16(128), 1e-6, pos0,
                          cache, cache.clone(), 32, 1e7)
    attention.attn_fwd(q, cache, cache, pos0, 4)
    attention.rms_norm(_bf16(3, 64), _bf16(64), 1e-6)
    attention.silu_mul(_bf16(3, 64))
    assert launches == ["gdn_attn_qk", "gdn_attn_fwd", "gdn_rms_norm", "gdn_silu_mul"]


def test_epilogue_and_decode_projection_launches(launches):
    epilogue.gated_rms_norm(_bf16(3, 128), _bf16(3, 128))
    linear.linear_decode(_bf16(3, 512), _bf16(8, 512))
    linear.gated_norm_linear_decode(_bf16(3, 512), _bf16(3, 512), None, 1e-6, 128, _bf16(8, 512))
    assert launches == ["gdn_gated_rmsnorm", "gdn_linear_decode", "gdn_linear_decode"]


def test_prepared_launches(launches):
    gated_delta.PreparedCall("gdn_x", (0,), {}, (), torch.device("cpu")).launch()
    chunked = gated_delta.PreparedChunked("gdn_chunk_fwd", (0,), {}, (), torch.device("cpu"))
    chunked.launch_prep()
    chunked.launch_scan(7)
    gated_delta.PreparedRecurrent(_lib.RecurrentArgs(), {}, torch.device("cpu")).launch(7)
    assert launches == ["gdn_x", "gdn_chunk_prep", "gdn_chunk_scan", "gdn_recurrent"]


def test_gated_delta_and_conv_launches(launches, monkeypatch):
    q, v = _bf16(1, 64, 1, 128), _bf16(1, 64, 1, 128)
    gates, par = _bf16(1, 64, 1), torch.zeros(1)
    state = torch.zeros(1, 1, 128, 128)
    for chunked in (False, True):
        gated_delta.gated_delta_update(q, q, v, gates, gates, par, par, state, chunked=chunked)
    qkv, w = _bf16(1, 64, 384), _bf16(384, 4)
    conv.gdn_conv_prologue(qkv, w, 1, 1, 128, 128)
    conv.gdn_conv_chunked(qkv, w, 1, 1, 128, 128, gates, gates, par, par)
    assert conv.gdn_conv_decode(qkv[:, :1], w, 1, 1, 128, 128, gates[:, :1], gates[:, :1], par, par, None, None)
    monkeypatch.setattr(conv, "_int_rows", lambda rows, n, dev, what: rows)
    conv.conv_state_commit(None, qkv[:, :4], torch.tensor([2], dtype=torch.int32))
    assert launches == ["gdn_recurrent", "gdn_chunk_fwd", "gdn_conv_prologue", "gdn_chunk_fwd_conv_masked",
                        "gdn_conv_decode", "gdn_conv_state_commit"]
