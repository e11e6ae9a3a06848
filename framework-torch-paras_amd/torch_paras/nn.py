"""Differentiable wrappers of the ``paras::`` fused ops, and the MoE layer.

``rms_norm``, ``swiglu`` and ``rotate_half`` keep the reference's signatures
(python/torch_paras/nn.py:75-89); their autograd nodes are C++ (csrc/torch/
ops_fused.cpp) and call the explicit backward ops.  ``moe_route`` / ``moe_ffn`` / ``moe_layer`` are this build's
additions (forward only).
"""
from __future__ import annotations

import torch

from . import _C  # (loading it registers the paras:: ops)

__all__ = ["rms_norm", "swiglu", "rotate_half", "moe_route", "moe_ffn", "moe_layer"]


def rms_norm(input: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    """Fused RMSNorm over the last dimension."""
    return _C.nn_rms_norm(input, weight, eps)


def swiglu(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """Fused ``silu(gate) * up``."""
    return _C.nn_swiglu(gate, up)


def rotate_half(x: torch.Tensor) -> torch.Tensor:
    """RoPE helper ``cat(-x2, x1)`` with ``x1, x2 = x.chunk(2, -1)``."""
    return _C.nn_rotate_half(x)


def moe_route(logits: torch.Tensor, k: int):
    """Top-k routing of ``logits [T, E]``: returns ``(topi [T,k] int64, topw [T,k]
    float32, order [T*k], inv_order [T*k], counts [E], offsets [E+1])`` --
    exactly what ``topk`` / ``softmax`` of the kept logits / stable ``argsort``
    of the expert ids / ``bincount`` / ``cumsum`` give."""
    return torch.ops.paras.moe_route(logits, k)


def moe_ffn(x, w_gate, w_up, w_down, topw, order, inv_order, offsets, k: int) -> torch.Tensor:
    """Grouped SwiGLU expert FFN over the routed rows plus the weighted combine."""
    return torch.ops.paras.moe_ffn(x, w_gate, w_up, w_down, topw, order, inv_order, offsets, k)


def moe_layer(x, router_logits, w_gate, w_up, w_down, k: int = 2) -> torch.Tensor:
    """One MoE layer: ``x [T,H]``, ``router_logits [T,E]``, ``w_gate/w_up [E,I,H]``,
    ``w_down [E,H,I]``."""
    return _C.nn_moe_layer(x, router_logits, w_gate, w_up, w_down, k)
