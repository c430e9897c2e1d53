"""A stack of dropout-linear layers with an activation between consecutive ones, as ONE autograd function whose
GEMM epilogues do the activation work.

The reference's models interleave exactly this (eval/mlp/model.py:31-40: DropoutMM, ReLU, DropoutMM, ..., DropoutMM;
eval/llm/model.py:62-66: DropoutMM, GELU, DropoutMM) as separate modules, i.e. one elementwise kernel per
activation in forward and one in backward, each a full pass over the hidden activations.  Here

    forward   h_{i+1} = act(s_i (keep_i ⊙ h_i) W_i^T)     the activation is applied to the fp32 accumulator in the
                                                            DSD kernel's store (sd_gemm_dsd_lists_act)
    backward  g_{i-1} = (s_i (g_i W_i) ⊙ keep_i) ⊙ act'     the derivative is multiplied in the SDD kernel's store
                                                            (sd_gemm_sdd_lists_actgrad); g_i is the gradient with
                                                            respect to layer i's pre-activation
              dW_i    = s_i g_i^T (keep_i ⊙ h_i)

so no activation kernel is launched in either direction.  ReLU's derivative is read off the activated tensor
(already kept as the next layer's input); GELU keeps the pre-activation as well.  The function and its
backward node are compiled (csrc/torch_bridge.cpp, ``mlp``).
"""
from __future__ import annotations

import torch

from ..hip import _loader
from ..hip.binding_gemm import _activation, _block_size
from .blockwise_dropout_matmul_hip import draw_source
from .tracing import traceable


@traceable
def blockwise_dropout_mlp(input: torch.Tensor, weights, block_size, p, activation: str | None = "relu",
                          masks=None, seed: int | None = None) -> torch.Tensor:
    """``W_n drop(act(... W_2 drop(act(W_1 drop(x))) ...))``: every layer drops blocks of its INPUT with
    probability p (a number, or one per layer; 0 keeps everything) and scales by 1/(1-p), ``activation``
    ("relu", "gelu" or None) sits between consecutive layers, none after the last.  ``masks`` (one bool mask per
    layer, True = dropped, or None where the layer draws one) pins the masks, ``seed`` pins the draws (layer i uses
    seed + i); otherwise they come from the device-resident generator.  ``input`` is [M, K], ``weights[i]`` is [out_i, in_i].

    With the device-resident generator a first layer with p = 0 whose input needs no gradient draws nothing (it runs as
    a dense product): the following layers then use the generator's draws 0, 1, ...; when the input does require a
    gradient that layer draws its (all kept) mask as well and the others use the draws 1, 2, ....  Results are valid
    either way; pass ``seed`` or ``masks`` where a run must not depend on it."""
    weights = list(weights)
    if not weights:
        raise ValueError("at least one layer is needed")
    ps = tuple(float(p) for _ in weights) if isinstance(p, (int, float)) else tuple(float(v) for v in p)
    if len(ps) != len(weights) or any(not 0 <= v < 1 for v in ps):
        raise ValueError("p must be one probability in [0, 1), or one per layer")
    if masks is not None and len(masks) != len(weights):
        raise ValueError("one mask per layer is needed")
    # the generator's state is made (a copy from the host) and reseeded when it is asked for: only where a mask is drawn
    draws = any(m is None for m in masks) if masks is not None else len(weights) > 1 or ps[0] > 0 or input.requires_grad
    return _loader.bridge().mlp(input, weights, _block_size(block_size), ps, _activation(activation),
                                None if masks is None else list(masks),
                                *(draw_source(input, seed) if draws else (None, None)))
