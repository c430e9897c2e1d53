"""Block-dropout matmul on the HIP kernels, as an autograd function.

Counterpart of the reference's ``BlockwiseDropoutMatmulCUDA``
(flash_dropout/functional/blockwise_dropout_matmul_cuda.py:7-59):

    forward   Y  = gemm_dsd(X, W, mask)            (:26)
    backward  dX = gemm_sdd(dY, W.T, mask)         (:46)
              dW = gemm_dsd(X.T, dY.T, mask.T).T   (:49-51)

Differences that matter to a caller: the kept-block lists are built once on the GPU in forward and
reused by both backward products (no per-iteration mask reads, no host sync); without a given mask
the Bernoulli draw happens inside the list-building launch; dW comes back as a contiguous [N, K]
tensor instead of a transposed view; bf16 works as well as fp16; shapes need not be multiples of
anything; block sizes that are multiples of 64 all run on the 64-block kernels; launches go to
torch's current stream.  The function and its backward node are compiled (csrc/torch_bridge.cpp,
``linear``): small layers are bound by the host, and the backward runs on autograd's thread
without the interpreter lock.  Under autocast the operands are cast to the autocast dtype
(the reference's ``custom_fwd(cast_inputs=torch.float16)``, :9); outside it they must already be
float16 / bfloat16.
"""
from __future__ import annotations

import torch

from ..hip import _loader
from ..hip.binding_gemm import GEMM, _block_size
from .tracing import traceable


def draw_source(like: torch.Tensor, seed: int | None):
    """(seed as an unsigned 64-bit number or None, generator state tensor or None): what a draw is made from."""
    if seed is not None:
        return int(seed) & (2 ** 64 - 1), None
    return None, (GEMM().rng_state(like.device) if like.is_cuda else None)


@traceable
def blockwise_dropout_matmul_mask(input: torch.Tensor, mask: torch.Tensor, block_size, p: float,
                                  weight: torch.Tensor) -> torch.Tensor:
    """Same as :func:`blockwise_dropout_matmul` with the mask given (True = dropped); argument order
    of the reference's naive counterpart (functional/naive.py:8-14)."""
    if not 0 <= p < 1:
        raise ValueError("Dropout probability must be in [0, 1)")
    return _loader.bridge().linear(input, weight, mask, _block_size(block_size), p, None, None)


@traceable
def blockwise_dropout_matmul(input: torch.Tensor, weight: torch.Tensor, block_size, p: float,
                             seed: int | None = None) -> torch.Tensor:
    """``(keep ⊙ input)/(1-p) @ weight.T`` with a fresh block mask (reference: …_cuda.py:56-59).

    The mask is drawn on the device inside the list-building launch; ``seed`` pins it (the same mask
    comes back from ``GEMM().random_lists(mask_shape, p, seed)``), otherwise it comes from the
    device-resident generator state, which starts at ``torch.initial_seed()`` and advances by one per
    call on the stream: nothing about the draw is a launch argument, so a captured graph draws a new
    mask at every replay."""
    if not 0 <= p < 1:
        raise ValueError("Dropout probability must be in [0, 1)")
    return _loader.bridge().linear(input, weight, None, _block_size(block_size), p, *draw_source(input, seed))
