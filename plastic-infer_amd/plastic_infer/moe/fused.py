"""Fused-MoE front end with the reference's signatures (src/plastic_infer/moe/fused.py).

  fused_topk                 :11-45   softmax over all experts -> top-k -> renormalise; fp32
                                      weights, int32 ids; rows >= num_token_non_padded get ids -1
  moe_align_block_size       :48-94   (sorted_token_ids, expert_ids, num_tokens_post_pad)
  fused_experts_impl         :169-273 routed gated-MLP FFN, result written over hidden_states
  fused_experts_decode_impl  :276-359 the same FFN into a new tensor
  FusedMoe                   :362-390 router + experts behind BaseMoeBackend
All run as HIP kernels. The permute plan orders routes inside an expert by ascending flattened
route index (deterministic; the reference's atomic-based order is not). Both FFN entry points
share one plan-driven native call (pia_moe_ffn): the plan of moe_align_block_size, the first expert
GEMM with the activation fused into its epilogue, the second with the routing weight, the sum; the
rounding points are the reference's (first GEMM output, activation output, second GEMM output
and the sum are each rounded to the storage dtype; with fp32 storage there is no rounding).
"""

from __future__ import annotations

import torch

from .. import _native as N
from ..kernel.moe_ops import moe_align_block_size as _align
from ..kernel.moe_ops import ACTIVATION_CODES, moe_topk
from .base import BaseMoeBackend

# Plan block of the expert GEMMs (the native call's own): the kernel takes 16 planned routes per work
# item, so the finest block wastes the fewest padded rows when an expert serves only a few routes.
EXPERT_BLOCK_M = 16


def fused_topk(hidden_states: torch.Tensor, gating_output: torch.Tensor, topk: int,
               renormalize: bool, num_token_non_padded: torch.Tensor | int | None = None
               ) -> tuple[torch.Tensor, torch.Tensor]:
    """(topk_weights fp32 [T, k], topk_ids int32 [T, k])."""
    assert hidden_states.shape[0] == gating_output.shape[0], "Number of tokens mismatch"
    N.require_device(gating_output, names=("gating_output",))
    n_np = None
    if num_token_non_padded is not None:
        n_np = int(num_token_non_padded.item()) if isinstance(num_token_non_padded, torch.Tensor) \
            else int(num_token_non_padded)
    return moe_topk(gating_output, topk, renormalize=renormalize, mode=0,
                    num_token_non_padded=n_np)


def moe_align_block_size(topk_ids: torch.Tensor, block_size: int, num_experts: int
                         ) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Pad each expert's route count to a multiple of block_size and lay routes out
    expert-contiguously. Sentinel = topk_ids.numel(); ids in [0, num_experts] are routed
    (num_experts itself is the extra sentinel expert of the fused-MoE convention)."""
    return _align(topk_ids, block_size, num_experts)


def _check_ffn_args(hidden_states, w1, w2, topk_weights, topk_ids, activation):
    assert hidden_states.dim() == 2 and w1.dim() == 3 and w2.dim() == 3
    assert hidden_states.shape[1] == w1.shape[2], "Hidden size mismatch"
    assert w1.shape[0] == w2.shape[0], "Expert cache size mismatch"
    assert w1.shape[1] == 2 * w2.shape[2], "Intermediate size mismatch"
    assert w2.shape[1] == hidden_states.shape[1], "Output hidden size mismatch"
    assert topk_weights.shape == topk_ids.shape, "topk shape mismatch"
    assert topk_ids.shape[0] == hidden_states.shape[0], "Number of tokens mismatch"
    assert hidden_states.is_contiguous(), "Hidden_states must be contiguous"
    assert w1.is_contiguous(), "Expert weights1 must be contiguous"
    assert w2.is_contiguous(), "Expert weights2 must be contiguous"
    if activation not in {"silu", "gelu", "gelu_tanh"}:
        raise ValueError(f"Unsupported activation: {activation}")
    if hidden_states.dtype not in (torch.bfloat16, torch.float16, torch.float32):
        raise NotImplementedError("expert GEMMs are built for bf16, fp16 and fp32 storage")
    assert w1.dtype == hidden_states.dtype and w2.dtype == hidden_states.dtype
    N.require_device(hidden_states, w1, w2, topk_weights, topk_ids,
                     names=("hidden_states", "w1", "w2", "topk_weights", "topk_ids"))


def routed_ffn_routes(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                      topk_weights: torch.Tensor, topk_ids: torch.Tensor,
                      route_out: torch.Tensor, activation: str = "silu",
                      apply_router_weight_on_input: bool = False,
                      act_buffer: torch.Tensor | None = None,
                      layer_experts: int | None = None) -> torch.Tensor:
    """The routed FFN of every route whose id is in [0, E), into route_out [T, k, H]: row
    (t, s) = w2[id] . act(w1[id] . x_t) times the routing weight, rounded to the storage dtype
    at the reference's points. Routes with id -1 are left untouched, so the routes of one
    token can be computed in several calls (e.g. experts already in HBM first, copied ones
    after their copies land) and summed once with moe_sum_reduce: the result is bit-identical
    to one call over all routes. act_buffer [T * k, I] may be shared between such calls.
    layer_experts: how many experts a layer has, where w1 and w2 are banks of more slots than that
    (the kernels' tiles are sized by it; such calls give the same one)."""
    M, H = hidden_states.shape
    E, two_i, _ = w1.shape
    k = topk_ids.shape[1]
    numel = M * k
    if numel == 0:
        return route_out
    if route_out.shape != (M, k, H) or not route_out.is_contiguous() \
            or route_out.dtype != hidden_states.dtype:
        raise ValueError(f"route_out must be a contiguous [{M}, {k}, {H}] tensor of the "
                         "hidden dtype")
    if act_buffer is not None and (
            act_buffer.dim() != 2 or act_buffer.stride(1) != 1 or act_buffer.shape[1] != two_i // 2
            or act_buffer.shape[0] < numel or act_buffer.dtype != hidden_states.dtype):
        raise ValueError(f"act_buffer must be [>= {numel}, {two_i // 2}] of the hidden dtype with "
                         "unit column stride")
    if hidden_states.stride(1) != 1 or hidden_states.shape[1] != w1.shape[2]:
        raise ValueError(f"hidden_states must be [T, {w1.shape[2]}] with contiguous rows")
    if w2.shape[1:] != (H, two_i // 2) or two_i % 2 \
            or not (w1.is_contiguous() and w2.is_contiguous()):
        raise ValueError("w1 must be contiguous [E, 2 I, H] and w2 contiguous [E, H, I]")
    if w1.dtype != hidden_states.dtype or w2.dtype != hidden_states.dtype:
        raise ValueError("hidden_states, w1 and w2 must share a dtype")
    if topk_weights.numel() != numel:
        raise ValueError("topk_weights must hold one weight per route")
    if topk_ids.numel() < numel:
        raise ValueError(f"topk_ids must hold the {numel} routes of hidden_states")
    N.require_device(hidden_states, w1, w2, topk_weights, topk_ids, route_out,
                     *(() if act_buffer is None else (act_buffer,)))
    E2 = w2.shape[0]
    if E2 < E:   # an expert without a second matrix gives zero rows, as any id of no weights does
        ids = topk_ids.reshape(-1)[:numel].view(M, k, 1)
        route_out.masked_fill_((ids >= E2) & (ids <= E), 0)
        w1 = w1[:E2]
    _ffn(hidden_states, w1, w2, topk_weights, topk_ids, activation, apply_router_weight_on_input,
         None, route_out, act_buffer, layer_experts)
    return route_out


def _ffn(hidden_states, w1, w2, topk_weights, topk_ids, activation, on_input, out, route_out=None,
         act_buffer=None, layer_experts=None) -> None:
    """The FFN of arguments already checked (pia_moe_ffn_bank), every buffer not given in one
    workspace."""
    act = ACTIVATION_CODES.get(activation)
    if act is None:
        raise ValueError(f"Unsupported activation: {activation}")
    M, H = hidden_states.shape
    E, inter, k = w1.shape[0], w2.shape[2], topk_ids.shape[1]
    ids = topk_ids.to(torch.int32).contiguous()
    weights = topk_weights.to(torch.float32).contiguous()
    dt, dev = N.dtype_code(hidden_states.dtype), hidden_states.device
    ws_bytes = N.query("pia_moe_ffn_workspace_bytes", M, k, E, H, inter, dt,
                       1 if act_buffer is None else 0, 1 if route_out is None else 0)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    N.call("pia_moe_ffn_bank", N.ptr(out), N.ptr(route_out), hidden_states.data_ptr(),
           hidden_states.stride(0), w1.data_ptr(), w2.data_ptr(), weights.data_ptr(),
           ids.data_ptr(), M, k, E, layer_experts or 0, H, inter, act, 1 if on_input else 0, dt,
           N.ptr(act_buffer), 0 if act_buffer is None else act_buffer.stride(0), ws.data_ptr(),
           ws_bytes, N.stream_of(dev))


def _routed_ffn(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                topk_weights: torch.Tensor, topk_ids: torch.Tensor, activation: str,
                apply_router_weight_on_input: bool, out: torch.Tensor,
                layer_experts: int | None) -> torch.Tensor:
    if topk_ids.numel():
        _ffn(hidden_states, w1, w2, topk_weights, topk_ids, activation,
             apply_router_weight_on_input, out, layer_experts=layer_experts)
    return out


def fused_experts_impl(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                       topk_weights: torch.Tensor, topk_ids: torch.Tensor,
                       activation: str = "silu",
                       apply_router_weight_on_input: bool = False,
                       layer_experts: int | None = None) -> torch.Tensor:
    """Returns ``hidden_states`` itself, overwritten with the routed output (the reference's
    contract: a caller that still needs the input must read it first or pass a copy).
    w1 [E, 2I, H] (gate rows then up rows), w2 [E, H, I]; ids in [0, E). layer_experts as for
    routed_ffn_routes."""
    _check_ffn_args(hidden_states, w1, w2, topk_weights, topk_ids, activation)
    return _routed_ffn(hidden_states, w1, w2, topk_weights, topk_ids, activation,
                       apply_router_weight_on_input, hidden_states, layer_experts)


def fused_experts_decode_impl(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                              topk_weights: torch.Tensor, topk_ids: torch.Tensor,
                              activation: str = "silu",
                              apply_router_weight_on_input: bool = False,
                              layer_experts: int | None = None) -> torch.Tensor:
    """The routed FFN into a new tensor (ids are expert or slot indices into w1 / w2).
    layer_experts as for routed_ffn_routes."""
    _check_ffn_args(hidden_states, w1, w2, topk_weights, topk_ids, activation)
    assert topk_weights.dtype == torch.float32
    assert topk_ids.dtype == torch.int32
    out = torch.empty_like(hidden_states)
    return _routed_ffn(hidden_states, w1, w2, topk_weights, topk_ids, activation,
                       apply_router_weight_on_input, out, layer_experts)


class FusedMoe(BaseMoeBackend):
    def forward(self, hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                gating_output: torch.Tensor, topk: int, renormalize: bool,
                activation: str = "silu",
                apply_router_weight_on_input: bool = False) -> torch.Tensor:
        topk_weights, topk_ids = fused_topk(hidden_states=hidden_states,
                                            gating_output=gating_output, topk=topk,
                                            renormalize=renormalize)
        return fused_experts_impl(hidden_states, w1, w2, topk_weights, topk_ids, activation,
                                  apply_router_weight_on_input=apply_router_weight_on_input,
                                  layer_experts=gating_output.shape[1])


__all__ = ["fused_topk", "moe_align_block_size", "fused_experts_impl",
           "fused_experts_decode_impl", "routed_ffn_routes", "FusedMoe", "EXPERT_BLOCK_M"]
