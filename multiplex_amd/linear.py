"""Decode-shape projections of the GatedDeltaNet mixer (``gdn_linear_decode``).

At decode a mixer layer's GEMMs have few rows (one token per batch row)
and are bound by reading their weights: in_proj's 12352 x 2048 and
out_proj's 2048 x 4096 bf16 matrices at hidden 2048 (``dflash.py:348-350,
377-378``).  ``gdn_linear_decode`` streams each weight once, split over
64-column tiles and 512-wide K slices, for 1..64 rows, and can fold the
epilogue's gated RMSNorm (``norm(out, z)``) into out_proj's operand load,
so the norm's output is never written.

Graph-replayed against the separate norm kernel plus hipBLASLt at hidden
2048, the fused norm + out_proj takes 7.4-8.1 us against 12.6-13.4 us up to
16 rows, and loses beyond (11.4 against 10.9 us at 32 rows, 16.4 against
13.1 us at 64).  So the mixer uses ``gated_norm_linear_decode`` up to
``FUSED_NORM_MAX_ROWS`` rows; ``linear_decode`` (the same call without the
norm) is the unfused reference for tests.  Up to 16 rows and above 2048
columns it runs ``gdn_linear_rows16``'s kernel, which leaves the workspace it
is given alone.

:func:`linear` is the layers' plain projection: a few rows by
``gdn_linear_rows16``, the library beyond.

The sliced kernel sums its K slices through a workspace of fp32 partials and one
ticket per output tile; the tickets must start at zero and every call
leaves them zero, so one zero-initialised workspace serves every call of a
module on one stream (calls that overlap, on several streams, need one
each).
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.autograd.forward_ad as forward_ad

from . import _lib
from .gated_delta import _dtype_code, _ptr, _require_device, _stream

__all__ = ["linear", "DECODE_MAX_ROWS", "FUSED_NORM_MAX_ROWS", "DecodeWorkspace", "linear_decode",
           "gated_norm_linear_decode", "linear_decode_workspace_bytes", "decode_shape_ok"]

DECODE_MAX_ROWS = 64
FUSED_NORM_MAX_ROWS = 16  # where the fused norm + projection beats the norm kernel plus the library GEMM
_K_SLICE = 512
_MAX_COLUMNS = 262144  # gdn_linear_rows16's limit


def linear_decode_workspace_bytes(M: int, N: int, K: int) -> int:
    return int(_lib.load().gdn_linear_decode_workspace_bytes(M, N, K))


def decode_shape_ok(M: int, N: int, K: int) -> bool:
    """Shapes ``gdn_linear_decode`` takes: 1..64 rows, K a multiple of 512, N of 8."""
    return 1 <= M <= DECODE_MAX_ROWS and K >= _K_SLICE and K % _K_SLICE == 0 and N % 8 == 0 and N > 0


class DecodeWorkspace:
    """A zero-initialised device buffer, grown (and zeroed again) on demand.

    Growing allocates, so a call under HIP graph capture must find the
    buffer already large enough: run the step once eagerly first.
    """

    def __init__(self):
        self.buf: Optional[torch.Tensor] = None

    def get(self, nbytes: int, device: torch.device) -> torch.Tensor:
        if self.buf is None or self.buf.device != device or self.buf.numel() < nbytes:
            self.buf = torch.zeros(nbytes, dtype=torch.uint8, device=device)
        return self.buf


def _rows(t: torch.Tensor, width: int, what: str) -> int:
    """Row stride (elements) of a ``[M, width]`` matrix with contiguous,
    16-byte aligned rows (e.g. a column slice of a wider buffer)."""
    if t.dim() != 2 or t.shape[1] != width or t.stride(1) != 1:
        raise ValueError(f"{what} must be [M, {width}] with contiguous rows")
    ld = t.stride(0) if t.shape[0] > 1 else width
    if ld < width or ld % 8 != 0 or t.data_ptr() % 16 != 0:
        raise ValueError(f"{what}: rows must be 16-byte aligned and a multiple of 8 elements apart")
    return int(ld)


def _launch(x, gate, norm_weight, eps, head_dim, weight, out, workspace):
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("gdn_linear_decode takes bf16 activations and weights")
    M, K = x.shape
    N = weight.shape[0]
    if weight.dim() != 2 or weight.shape[1] != K or not weight.is_contiguous():
        raise ValueError(f"weight must be a contiguous [N, {K}] matrix")
    if not decode_shape_ok(M, N, K):
        raise ValueError(f"gdn_linear_decode takes 1..{DECODE_MAX_ROWS} rows, K a multiple of 512 and N of 8 "
                         f"(got M={M}, N={N}, K={K})")
    dev = _require_device([x, gate, norm_weight, weight, out], ["x", "gate", "norm_weight", "weight", "out"])
    ldx = _rows(x, K, "x")
    ldg = _rows(gate, K, "gate") if gate is not None else 0
    if out is None:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    ldo = _rows(out, N, "out")
    need = linear_decode_workspace_bytes(M, N, K)
    ws = (workspace if workspace is not None else DecodeWorkspace()).get(need, dev)
    nw_dt = _dtype_code(norm_weight, "norm_weight") if norm_weight is not None else 0
    _lib.call(dev, "gdn_linear_decode", _ptr(x), ldx, _ptr(gate), ldg, _ptr(norm_weight), nw_dt, float(eps),
              int(head_dim), _ptr(weight), _ptr(out), ldo, M, N, K, _ptr(ws), ws.numel(), _stream(dev))
    return out


def linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``x @ weight.T`` (``torch.nn.functional.linear`` without a bias).

    A few rows of bf16 (:func:`_rows16_shape` has the sizes) by
    ``gdn_linear_rows16``; the library elsewhere, and where differentiation,
    autocast, a function transform or a tensor subclass needs its operator.
    The call costs the host 6.7 us, the library's 17.6.
    """
    N, K = weight.shape
    rows = x.numel() // K if K else 0
    if (_rows16_shape(rows, N, K) and x.dtype is torch.bfloat16 and weight.dtype is torch.bfloat16
            and x.is_cuda and weight.is_cuda and x.shape[-1] == K and not _needs_operator(x, weight)
            and x.is_contiguous() and weight.is_contiguous() and x.get_device() == weight.get_device()):
        xp, wp = x.data_ptr(), weight.data_ptr()
        if (xp | wp) % 16 == 0:
            return _rows16(x, xp, wp, rows, N, K)
    return torch.nn.functional.linear(x, weight)


_transform_level = getattr(torch._C._functorch, "maybe_current_level", None)
_dispatch_modes = getattr(torch._C, "_len_torch_dispatch_stack", None)


def _needs_operator(x, weight) -> bool:
    """Whether something follows or replaces the operator on these operands: a
    recorded gradient, a forward-mode tangent (its tensors are plain ones that
    ask for no gradient), a function transform (vmap, jvp, grad), a dispatch
    mode or a trace, autocast, a tensor subclass."""
    if (type(x) is not torch.Tensor or type(weight) not in (torch.Tensor, torch.nn.Parameter)
            or torch.is_autocast_enabled() or (torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad))):
        return True
    if _transform_level is None or _transform_level() is not None:
        return True
    if _dispatch_modes is None or _dispatch_modes() or torch.jit.is_tracing():
        return True
    # (outside a dual level, -1, no tensor has a tangent)
    return getattr(forward_ad, "_current_level", 0) >= 0 and any(
        forward_ad.unpack_dual(t).tangent is not None for t in (x, weight))


def _rows16_shape(rows, N, K) -> bool:
    """The sizes :func:`linear` gives to ``gdn_linear_rows16`` (which refuses
    more than ``_MAX_COLUMNS`` columns).

    The lines follow graph-replayed times with the weights read from memory,
    as those of a model's layers are (each call another of 600 MB of them);
    behind them, after the slash, calls of one weight that stays in the
    last-level cache, where the library gains more.  us, against the library's:
      K to 4096, 16 rows:  4096 x 4096 9.9 / 9.3, 14.7 / 11.6 (4 rows 8.0 / 7.3, 14.7 / 11.3);
        10240 x 4096 18.4 / 16.8, 25.0 / 19.6; 12352 x 2048 12.2 / 11.5, 15.1 / 10.8 (8 rows 11.4 / 10.7,
        15.1 / 10.8); 6144 x 4096 13.6 / 12.9, 14.4 / 11.3.  Of 120 sizes from 512 to 4096 by 2056 to 24576
        it is the slower one at 13, by 10% at most (K = 2560 and 3584 at 4608 to 8192 columns, 16384 columns);
        with the weight in the cache at 75, by 57% at most (K = 2560 at 4608 to 6144 columns)
      K to 8192, 4 rows:   4096 x 8192 15.5 / 12.4, 15.5 / 13.0; 12288 x 8192 35.3 / 29.6, 39.5 / 31.4
      K to 12288, 2 rows:  4096 x 12288 18.4 / 16.2, 21.0 / 17.0; 16384 x 12288 69.9 / 69.1, 82.4 / 86.4
      K over 4096 at 4104 to 8192 columns, where the busiest CU has two 16-column tiles and most have
        fewer, is the library's: 5120 x 5120 at 4 rows 14.5 / 13.0, 14.0 / 11.5; 6144 x 8192 23.2 / 19.3,
        21.4 / 17.9 (and, with two on every CU, 8192 x 8192 32.0 / 20.3, 28.9 / 21.7; 8192 x 6144, 21% faster
        than the library from memory, goes there with them)
    """
    if K <= 4096:
        most = 16
    elif 4096 < N <= 8192:
        most = 0
    else:
        most = 4 if K <= 8192 else 2
    return 1 <= rows <= most and 512 <= K <= 12288 and K % _K_SLICE == 0 and 2048 < N <= _MAX_COLUMNS and N % 8 == 0


def _rows16(x, x_addr, w_addr, rows, N, K):
    dev = x.device
    out = torch.empty(*x.shape[:-1], N, dtype=torch.bfloat16, device=dev)
    _lib.call(dev, "gdn_linear_rows16", x_addr, K, w_addr, out.data_ptr(), N, rows, N, K, _stream(dev))
    return out


def linear_decode(x: torch.Tensor, weight: torch.Tensor, *, out: Optional[torch.Tensor] = None,
                  workspace: Optional[DecodeWorkspace] = None) -> torch.Tensor:
    """``x @ weight.T`` for ``x [M <= 64, K]`` (rows may be a column slice)."""
    return _launch(x, None, None, 0.0, 0, weight, out, workspace)


def gated_norm_linear_decode(y: torch.Tensor, z: torch.Tensor, norm_weight: Optional[torch.Tensor], eps: float,
                             head_dim: int, weight: torch.Tensor, *, out: Optional[torch.Tensor] = None,
                             workspace: Optional[DecodeWorkspace] = None) -> torch.Tensor:
    """``gated_rms_norm(y, z, norm_weight, eps) @ weight.T`` per head of
    ``head_dim`` (64 or 128) columns, with the norm computed inside the
    projection's operand load (gdn_gated_rmsnorm's rounding points).
    y, z ``[M, K]``."""
    if z.dtype != torch.bfloat16:
        raise ValueError("z must be bf16")
    if norm_weight is not None:
        if tuple(norm_weight.shape) != (head_dim,):
            raise ValueError(f"norm_weight must be [{head_dim}]")
        norm_weight = norm_weight.contiguous()
    return _launch(y, z, norm_weight, eps, head_dim, weight, out, workspace)
