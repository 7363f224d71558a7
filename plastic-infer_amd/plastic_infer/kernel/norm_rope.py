"""RMSNorm and per-head RMSNorm + RoPE of a decode step, one launch each.

The formulas of exec.attention's rms_norm and RoPE helpers (reference:
src/plastic_infer/exec/attention.py:53-95) with fp32 arithmetic and one rounding of the result.
Tensors the kernels do not take (dtypes that differ, non-contiguous rows, values that autograd
follows: the kernels record nothing for it) go through those helpers.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from .. import _native as N

EPS = 1e-5   # of the reference's rms_norm


def _fits(*tensors: torch.Tensor) -> bool:
    """Contiguous device tensors of one dtype that the kernels are built for, with no derivative
    to be taken of them in either mode (inside a dual level any of them may carry a tangent)."""
    if getattr(forward_ad, "_current_level", -1) >= 0:
        return False
    dt, dev, grad = tensors[0].dtype, tensors[0].device, torch.is_grad_enabled()
    for t in tensors:
        if t.dtype != dt or not t.is_contiguous() or t.device != dev or (grad and t.requires_grad):
            return False
    return dev.type == "cuda" and dt in (torch.bfloat16, torch.float16, torch.float32)


def _plain(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt(torch.mean(x * x, dim=-1, keepdim=True) + EPS) * weight


def rms_norm_rows(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """RMSNorm over the last dimension."""
    n = x.shape[-1]
    if n == 0 or weight.shape != (n,) or not _fits(x, weight):
        return _plain(x, weight)
    out = torch.empty_like(x)
    N.call("pia_rms_norm", out.data_ptr(), None, x.data_ptr(), None, weight.data_ptr(),
           x.numel() // n, n, EPS, N.dtype_code(x.dtype), N.stream_of(x.device))
    return out


def add_rms_norm_rows(x: torch.Tensor, y: torch.Tensor, weight: torch.Tensor
                      ) -> tuple[torch.Tensor, torch.Tensor]:
    """(x + y, its RMSNorm)."""
    n = x.shape[-1]
    if n == 0 or weight.shape != (n,) or y.shape != x.shape or not _fits(x, y, weight):
        s = x + y
        return s, rms_norm_rows(s, weight)
    s, out = torch.empty_like(x), torch.empty_like(x)
    N.call("pia_rms_norm", out.data_ptr(), s.data_ptr(), x.data_ptr(), y.data_ptr(),
           weight.data_ptr(), x.numel() // n, n, EPS, N.dtype_code(x.dtype),
           N.stream_of(x.device))
    return s, out


def _rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    x1, x2 = x.chunk(2, dim=-1)
    return x * cos[:, None, :] + torch.cat([-x2, x1], dim=-1) * sin[:, None, :]


def qk_norm_rope(q: torch.Tensor, k: torch.Tensor, q_weight: torch.Tensor | None,
                 k_weight: torch.Tensor | None, cos: torch.Tensor, sin: torch.Tensor
                 ) -> tuple[torch.Tensor, torch.Tensor]:
    """q [B, Hq, D] and k [B, Hkv, D]: RMSNorm over D by the weights (None: no norm), then the
    rotate-half RoPE by each row's own table rows cos, sin [B, D]. Contiguous results."""
    B, Hq, D = q.shape
    Hkv = k.shape[1]
    norm = q_weight is not None
    ws = (q_weight, k_weight) if norm else ()
    if D == 0 or D % 2 or k.shape != (B, Hkv, D) or cos.shape != (B, D) or sin.shape != (B, D) \
            or any(w.shape != (D,) for w in ws) or not _fits(q, k, cos, sin, *ws):
        if norm:
            q, k = _plain(q, q_weight), _plain(k, k_weight)
        return _rope(q, cos, sin).contiguous(), _rope(k, cos, sin).contiguous()
    qo, ko = torch.empty_like(q), torch.empty_like(k)
    N.call("pia_qk_norm_rope", qo.data_ptr(), ko.data_ptr(), q.data_ptr(), k.data_ptr(),
           N.ptr(q_weight), N.ptr(k_weight), cos.data_ptr(), sin.data_ptr(), B, Hq, Hkv, D, EPS,
           N.dtype_code(q.dtype), N.stream_of(q.device))
    return qo, ko


__all__ = ["rms_norm_rows", "add_rms_norm_rows", "qk_norm_rope"]
