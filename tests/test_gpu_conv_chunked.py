"""GPU checks of the mixer prefill with the conv prologue fused into the
chunked prep (``gdn_conv_chunked`` / ``gdn_chunk_fwd_conv``).

The fused prep forms q, k and v with the conv prologue's arithmetic, so y,
the state and the new conv state must equal ``gdn_conv_prologue`` followed
by ``gated_delta_update(..., chunked=True)`` bit for bit; that pair is
itself checked against the oracle in ``tests/test_gpu_configs.py`` and
``tests/test_gpu_prologue.py``.  Cases: the benchmark's T=4096 prefill at
full width (also against the oracle on head subsets), equal-length rows with
a partial last chunk, packed sequences with lengths below the conv window
(0, 1, 2 tokens) next to long ones, fp32 taps, GQA groups of 1 and 3, qkv
and gates read as column slices of one buffer, pooled states, and rows of
no tokens.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import multiplex_amd as mx
from gdn_cases import STATE_TOL, Y_TOL, head_errs_state, rel_err, row_errs_y
from oracle import gdn

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def _inputs(seed, B, S, Hk, Hv, *, cs=True, state=True, w_dtype=torch.bfloat16, n_seqs=None):
    gen = torch.Generator().manual_seed(seed)
    C = 2 * Hk * D + Hv * D
    n = B if n_seqs is None else n_seqs
    t = dict(
        qkv=torch.randn(B, S, C, generator=gen).to(torch.bfloat16),
        w=(torch.randn(C, 4, generator=gen) * 0.3).to(w_dtype),
        a=torch.randn(B, S, Hv, generator=gen).to(torch.bfloat16),
        b=torch.randn(B, S, Hv, generator=gen).to(torch.bfloat16),
        A_log=torch.rand(Hv, generator=gen) * math.log(16.0),
        dt_bias=torch.rand(Hv, generator=gen) * 2 - 1,
        cs=(torch.randn(n, 3, C, generator=gen) * 0.5).to(torch.bfloat16) if cs else None,
        state=(torch.randn(n, Hv, D, D, generator=gen) * 0.02) if state else None,
    )
    return {k: (None if v is None else v.to(DEV)) for k, v in t.items()}


def _unfused(t, Hk, Hv, cu=None, state_index=None, pool=None):
    q, k, v, cs = mx.gdn_conv_prologue(t["qkv"], t["w"], Hk, Hv, D, D, t["cs"], cu_seqlens=cu)
    st = pool if pool is not None else t["state"]
    y, s = mx.gated_delta_update(q, k, v, t["a"], t["b"], t["A_log"], t["dt_bias"], st, cu_seqlens=cu,
                                 chunked=True, state_index=state_index)
    return y, s, cs, (q, k, v)


def _fused(t, Hk, Hv, cu=None, state_index=None, pool=None):
    st = pool if pool is not None else t["state"]
    return mx.gdn_conv_chunked(t["qkv"], t["w"], Hk, Hv, D, D, t["a"], t["b"], t["A_log"], t["dt_bias"], st,
                               t["cs"], cu_seqlens=cu, state_index=state_index)


def _assert_equal(fused, unfused):
    y, s, cs = fused
    y2, s2, cs2 = unfused[:3]
    torch.cuda.synchronize()
    assert torch.equal(y, y2), "y differs from the unfused pair"
    assert torch.equal(s, s2), "state differs from the unfused pair"
    assert torch.equal(cs, cs2), "conv state differs from the unfused pair"


def _np(t):
    return t.detach().double().cpu().numpy()


def test_t4096_full_width_equals_unfused_and_oracle():
    Hk, Hv, T = 16, 32, 4096
    t = _inputs(2001, 1, T, Hk, Hv)
    fused = _fused(t, Hk, Hv)
    unfused = _unfused(t, Hk, Hv)
    _assert_equal(fused, unfused)
    # the oracle on a subset of heads, from the raw qkv
    hks, heads = [0, 15], [0, 1, 30, 31]
    ch = np.concatenate([np.arange(h * D, (h + 1) * D) for h in hks]
                        + [np.arange((Hk + h) * D, (Hk + h + 1) * D) for h in hks]
                        + [np.arange((2 * Hk + h) * D, (2 * Hk + h + 1) * D) for h in heads])
    qr, kr, vr, csr, _ = gdn.conv_prologue(_np(t["qkv"])[:, :, ch], _np(t["w"])[ch], len(hks), len(heads), D, D,
                                           _np(t["cs"])[:, :, ch])
    np.testing.assert_array_equal(fused[2].float().cpu().numpy()[:, :, ch], csr)
    g = gdn.compute_g(_np(t["A_log"])[heads], _np(t["a"])[:, :, heads], _np(t["dt_bias"])[heads])
    beta = gdn.compute_beta(_np(t["b"])[:, :, heads])
    # the kernel's bf16 q, k, v (bit-equal to the unfused prologue's) feed the recurrent oracle
    q, k, v = unfused[3]
    y_ref, s_ref = gdn.recurrent(_np(q[:, :, hks]), _np(k[:, :, hks]), _np(v[:, :, heads]), g, beta,
                                 _np(t["state"])[:, heads])
    assert rel_err(q[:, :, hks].float().cpu().numpy(), qr) <= Y_TOL
    assert rel_err(v[:, :, heads].float().cpu().numpy(), vr) <= Y_TOL
    assert row_errs_y(fused[0][:, :, heads].float().cpu().numpy(), y_ref).max() <= Y_TOL
    assert head_errs_state(fused[1][:, heads].cpu().numpy(), s_ref).max() <= STATE_TOL


@pytest.mark.parametrize("Hk,Hv,w_dtype", [(2, 4, torch.bfloat16), (2, 2, torch.float32), (1, 3, torch.bfloat16)])
def test_rows_with_a_partial_chunk_equal_unfused(Hk, Hv, w_dtype):
    t = _inputs(2002 + Hv, 2, 200, Hk, Hv, w_dtype=w_dtype)
    _assert_equal(_fused(t, Hk, Hv), _unfused(t, Hk, Hv))


@pytest.mark.parametrize("Hk,Hv,w_dtype", [(16, 32, torch.bfloat16), (16, 32, torch.float32), (8, 32, torch.bfloat16)])
def test_head_pairs_equal_single_heads(Hk, Hv, w_dtype):
    """737 tokens of 32 heads take two v-heads a prep workgroup; the same rows as one packed sequence take
    one.  The same arithmetic per head, so the same bits, fused and from q, k and v with and without a mask."""
    T = 737
    t = _inputs(2003 + Hk, 1, T, Hk, Hv, w_dtype=w_dtype)
    _assert_equal(_fused(t, Hk, Hv), _fused(t, Hk, Hv, cu=[0, T]))
    q, k, v, _ = mx.gdn_conv_prologue(t["qkv"], t["w"], Hk, Hv, D, D, t["cs"])
    mask = torch.rand(1, T, generator=torch.Generator().manual_seed(5)) < 0.8
    for m in (None, mask.to(DEV)):
        args = (q, k, v, t["a"], t["b"], t["A_log"], t["dt_bias"], t["state"], m)
        for x, y in zip(mx.gated_delta_update(*args), mx.gated_delta_update(*args, cu_seqlens=[0, T])):
            assert torch.equal(x, y)


@pytest.mark.parametrize("with_cs", [True, False])
def test_packed_short_and_empty_sequences_equal_unfused(with_cs):
    """Lengths 2, 0, 68, 130, 1, 3: conv windows reaching into the conv
    state, an empty sequence (its conv state passes through), chunk edges."""
    Hk, Hv = 2, 4
    lens = [2, 0, 68, 130, 1, 3]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = _inputs(2010, 1, int(cu[-1]), Hk, Hv, cs=with_cs, n_seqs=len(lens))
    for cu_arg in (cu.tolist(), torch.tensor(cu, device=DEV)):
        _assert_equal(_fused(t, Hk, Hv, cu=cu_arg), _unfused(t, Hk, Hv, cu=cu_arg))


def test_column_slices_of_one_projection_buffer():
    """qkv, a and b as column slices of one fused in_proj output."""
    Hk, Hv, S = 2, 4, 150
    t = _inputs(2020, 2, S, Hk, Hv)
    C = t["qkv"].shape[-1]
    buf = torch.zeros(2, S, C + 64 + 2 * Hv, dtype=torch.bfloat16, device=DEV)
    buf[..., :C] = t["qkv"]
    buf[..., C + 64:C + 64 + Hv] = t["a"]
    buf[..., C + 64 + Hv:] = t["b"]
    sl = dict(t, qkv=buf[..., :C], a=buf[..., C + 64:C + 64 + Hv], b=buf[..., C + 64 + Hv:])
    _assert_equal(_fused(sl, Hk, Hv), _unfused(t, Hk, Hv))


def test_pooled_states_equal_unfused():
    Hk, Hv = 2, 4
    lens = [70, 5, 130]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = _inputs(2030, 1, int(cu[-1]), Hk, Hv, n_seqs=len(lens))
    gen = torch.Generator().manual_seed(2031)
    pool = (torch.randn(6, Hv, D, D, generator=gen) * 0.02).to(DEV)
    idx = torch.tensor([4, 0, 2], dtype=torch.int32, device=DEV)
    p1, p2 = pool.clone(), pool.clone()
    y, _, cs = _fused(t, Hk, Hv, cu=cu.tolist(), state_index=idx, pool=p1)
    y2, _, cs2, _ = _unfused(t, Hk, Hv, cu=cu.tolist(), state_index=idx, pool=p2)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(cs, cs2)
    assert torch.equal(p1, p2)


def test_rows_of_no_tokens_pass_the_conv_state_through():
    Hk, Hv = 2, 4
    t = _inputs(2040, 3, 0, Hk, Hv)
    y, s, cs = _fused(t, Hk, Hv)
    torch.cuda.synchronize()
    assert y.shape == (3, 0, Hv, D)
    assert torch.equal(cs, t["cs"])
    assert torch.equal(s, t["state"])


def test_mixer_prefill_takes_the_fused_path_and_matches_unfused():
    """The mixer's chunked prefill (fused) against the same layer with the
    prologue launched on its own."""
    m = mx.GatedDeltaNet(256, 2, 4, D, D, device=DEV)
    m.reset_parameters(torch.Generator().manual_seed(2050))
    x = torch.randn(2, 100, 256, generator=torch.Generator().manual_seed(2051)).to(torch.bfloat16).to(DEV)
    with torch.no_grad():
        c1, c2 = mx.ArraysCache(), mx.ArraysCache()
        assert m._fused_prefill(m._project(x)[0], None)
        out1 = m(x, None, c1)
        fused = m._fused_prefill
        m._fused_prefill = lambda qkv, mask: False
        try:
            out2 = m(x, None, c2)
        finally:
            m._fused_prefill = fused
        torch.cuda.synchronize()
    assert torch.equal(out1, out2)
    assert torch.equal(c1[0], c2[0]) and torch.equal(c1[1], c2[1])


@pytest.mark.parametrize("B,S,Hk,Hv,w_dtype,kind", [
    (4, 301, 2, 4, torch.bfloat16, "left_pad"),
    (2, 129, 1, 3, torch.float32, "random"),
    (1, 64, 2, 2, torch.bfloat16, "whole_row"),
    (2, 1000, 16, 32, torch.bfloat16, "random"),  # head pairs
    (1, 737, 16, 32, torch.float32, "left_pad"),
])
@pytest.mark.parametrize("with_cs", [True, False])
def test_masked_rows_equal_unfused(B, S, Hk, Hv, w_dtype, kind, with_cs):
    """A mask given to the fused pass and to the two launches: the same bits, and masked rows that hold NaN
    and inf reach neither (left pads, single tokens at chunk edges and in the conv windows, a whole row)."""
    t = _inputs(2060 + S, B, S, Hk, Hv, cs=with_cs, w_dtype=w_dtype)
    gen = torch.Generator().manual_seed(S)
    if kind == "left_pad":
        pad = torch.randint(0, S, (B, 1), generator=gen)
        mask = torch.arange(S)[None, :] >= pad
    else:
        mask = torch.rand(B, S, generator=gen) < (0.7 if kind == "random" else 0.0)
    mask = mask.to(DEV)
    t["qkv"][~mask] = float("nan")
    t["qkv"][:, ::3][~mask[:, ::3]] = float("inf")
    q, k, v, cs = mx.gdn_conv_prologue(t["qkv"], t["w"], Hk, Hv, D, D, t["cs"], mask)
    y, s = mx.gated_delta_update(q, k, v, t["a"], t["b"], t["A_log"], t["dt_bias"], t["state"], mask, chunked=True)
    got = mx.gdn_conv_chunked(t["qkv"], t["w"], Hk, Hv, D, D, t["a"], t["b"], t["A_log"], t["dt_bias"], t["state"],
                              t["cs"], mask=mask)
    _assert_equal(got, (y, s, cs))
    assert torch.isfinite(got[0].float()).all() and torch.isfinite(got[1]).all()


def _masked_pair(t, Hk, Hv, mask, cu, idx=None, pools=(None, None)):
    """The fused pass and the two launches on the same masked rows."""
    q, k, v, cs = mx.gdn_conv_prologue(t["qkv"], t["w"], Hk, Hv, D, D, t["cs"], mask, cu_seqlens=cu)
    y, s = mx.gated_delta_update(q, k, v, t["a"], t["b"], t["A_log"], t["dt_bias"],
                                 t["state"] if idx is None else pools[1], mask, cu_seqlens=cu, chunked=True,
                                 state_index=idx)
    got = mx.gdn_conv_chunked(t["qkv"], t["w"], Hk, Hv, D, D, t["a"], t["b"], t["A_log"], t["dt_bias"],
                              t["state"] if idx is None else pools[0], t["cs"], cu_seqlens=cu, state_index=idx,
                              mask=mask)
    return got, (y, s, cs)


@pytest.mark.parametrize("with_cs", [True, False])
@pytest.mark.parametrize("pooled", [False, True])
@pytest.mark.parametrize("packed", [True, False])
def test_masked_packed_and_pooled_rows_equal_unfused(packed, pooled, with_cs):
    """A mask with packed sequences (lengths below the conv window and none at all among them, their first
    and last tokens masked), with pooled states, and with both."""
    Hk, Hv = 2, 4
    lens = [2, 0, 68, 130, 1, 3] if packed else [150] * 3
    n, total = len(lens), sum(lens)
    at = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = _inputs(2080, 1 if packed else n, total if packed else 150, Hk, Hv, cs=with_cs, n_seqs=n)
    gen = torch.Generator().manual_seed(2081)
    mask = torch.rand(total, generator=gen) < 0.7
    for start, length in zip(at, lens):
        if length > 2:
            mask[[start, start + length - 1]] = False
    mask = mask.view(t["qkv"].shape[:2]).to(DEV)
    t["qkv"][~mask] = float("nan")
    pool = (torch.randn(8, Hv, D, D, generator=gen) * 0.02).to(DEV)
    idx = torch.tensor([4, 0, 2, 7, 1, 6][:n], dtype=torch.int32, device=DEV) if pooled else None
    pools = (pool.clone(), pool.clone())
    got, want = _masked_pair(t, Hk, Hv, mask, at.tolist() if packed else None, idx, pools)
    _assert_equal(got, want)
    assert torch.isfinite(got[0].float()).all() and torch.isfinite(got[1]).all()
    if pooled:
        left = [i for i in range(8) if i not in idx.tolist()]
        assert torch.equal(pools[0][left], pool[left])


@pytest.mark.parametrize("pooled", [False, True])
def test_mixer_masked_prefill_takes_the_fused_path_and_matches_unfused(pooled):
    """The layer on left-padded prompts, with dense and with pooled states, against the same layer with the
    prologue launched on its own."""
    m = mx.GatedDeltaNet(256, 2, 4, D, D, device=DEV)
    m.reset_parameters(torch.Generator().manual_seed(2090))
    gen = torch.Generator().manual_seed(2091)
    x = torch.randn(3, 100, 256, generator=gen).to(torch.bfloat16).to(DEV)
    mask = (torch.arange(100)[None, :] >= torch.tensor([[0], [37], [98]])).to(DEV)
    cs = torch.randn(3, 3, m.conv_dim, generator=gen).to(torch.bfloat16).to(DEV)
    states = (torch.randn(3, 4, D, D, generator=gen) * 0.02).to(DEV)
    outs = []
    with torch.no_grad():
        for fused in (True, False):
            c = mx.ArraysCache()
            c[0] = cs.clone()
            if pooled:
                pool = mx.StatePool(5, 4, D, D, device=DEV)
                slots = pool.alloc(5)
                pool.release(slots[:1] + slots[3:4])
                c[1] = mx.PooledBatch(pool, [slots[i] for i in (4, 1, 2)])
                pool.scatter(c[1].slots, states)
            else:
                c[1] = states.clone()
            if fused:
                assert m._fused_prefill(m._project(x)[0], mask)
            else:
                m._fused_prefill = lambda qkv, mask: False
            y = m(x, mask, c)
            outs.append((y, c[1].pool.gather(c[1].slots) if pooled else c[1], c[0]))
    _assert_equal(*outs)
