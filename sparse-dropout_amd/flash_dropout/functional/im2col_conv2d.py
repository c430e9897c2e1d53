"""2-D convolution as im2col + matmul, dense and with block dropout on the patch matrix.

Reference: flash_dropout/functional/im2col_conv2d.py:5-27 — ``F.unfold`` to (N, C*R*S, P*Q), permute
to (N, P*Q, C*R*S), ``F.linear`` with ``kernel.view(K, -1)``, back to (N, K, P, Q).  Here the patch
matrix [N*P*Q, C*R*S] (same column order c*R*S + r*S + s) is produced by the HIP gather kernel and
multiplied by the HIP GEMMs; the result is returned, like the reference's, as an (N, K, P, Q) view
of an (N, P*Q, K) buffer.

The block-dropout variant is the one the reference left as comments in its conv layer
(flash_dropout/layers/dropout_conv.py:86-99): one Bernoulli per block_size x block_size tile of the
patch matrix; dropped tiles are neither gathered nor multiplied.
"""
from __future__ import annotations

from math import ceil

import torch
import torch.nn.functional as F

from ..hip import _loader
from ..hip.binding_gemm import GEMM, _block_size
from .blockwise_dropout_matmul_hip import draw_source
from .tracing import traceable


# Let the forward run without a patch matrix (sd_conv2d_taps_forward or sd_conv2d_dsd_lists).  Module-level switch so that tests and
# benchmarks can compare both routes: off, the forward goes through the matrix; on, where the library takes the geometry and,
# with a mask, where that is expected to be faster (few rows and pointwise kernels of planes go through the matrix all the same).
IMPLICIT_FORWARD = True
# The same for the input gradient in one launch (sd_conv2d_taps_dx or sd_conv2d_dx_blocks): on, masked layers whose matrix is wider than a
# block, at most 256 MB and folded fast make the gradient of the patch matrix all the same.  (Products run tap by tap when both
# switches are on.)
FUSED_INPUT_GRADIENT = True

_ROUTES = (None, "implicit", "fused", "explicit")


def conv_last_routes() -> dict:
    """{"forward": ..., "dx": ..., "dw": ...} of the process's last convolution run through this module: "implicit" /
    "fused" (no patch matrix in memory: sd_conv2d_taps_*, or sd_conv2d_dsd_lists, sd_conv2d_dw_lists, sd_conv2d_dx_blocks) or "explicit"
    (the patch matrix or its gradient in memory around the GEMMs: the library does not take the geometry, a switch above
    is off, or, with a mask, that is expected to be faster); None for a product that was not computed.  Nothing falls back
    to the patch matrix unseen."""
    return {k: _ROUTES[v] for k, v in zip(("forward", "dx", "dw"), _loader.bridge().conv_routes())}


def _pair(v) -> tuple[int, int]:
    if isinstance(v, int):
        return (v, v)
    a, b = v
    return (int(a), int(b))


def _conv2d(input, kernel, mask, block_size, p, padding, stride, dilation, draw=(None, None)):
    return _loader.bridge().conv2d(input, kernel, mask, block_size, p, _pair(padding), _pair(stride), _pair(dilation),
                                   *draw, IMPLICIT_FORWARD, FUSED_INPUT_GRADIENT)


@traceable
def im2col_conv2d(input: torch.Tensor, kernel: torch.Tensor, padding=(0, 0), stride=(1, 1),
                  dilation=(1, 1)) -> torch.Tensor:
    """Dense convolution through the patch matrix (reference: im2col_conv2d.py:5-27)."""
    return _conv2d(input, kernel, None, 0, 0.0, padding, stride, dilation)


def conv_patch_matrix_shape(input_shape, kernel_shape, padding=(0, 0), stride=(1, 1), dilation=(1, 1)):
    """(N*P*Q, C*R*S): the matrix the block mask of the conv variant is drawn over."""
    n, c, h, w = input_shape
    _, _, r, s = kernel_shape
    po, qo = GEMM.conv_out_hw(h, w, r, s, _pair(padding), _pair(stride), _pair(dilation))
    return n * po * qo, c * r * s


@traceable
def blockwise_dropout_conv2d_mask(input, mask, block_size, p: float, kernel, padding=(0, 0),
                                  stride=(1, 1), dilation=(1, 1)) -> torch.Tensor:
    """Block-dropout convolution with the mask given: ``mask`` is bool
    [ceil(N*P*Q/bs), ceil(C*R*S/bs)], True = dropped."""
    if not 0 <= p < 1:
        raise ValueError("Dropout probability must be in [0, 1)")
    bs = _block_size(block_size)
    if bs % 64:
        raise NotImplementedError(f"block_size {bs}: the convolution takes multiples of 64 (the matmul also 32)")
    return _conv2d(input, kernel, mask, bs, p, padding, stride, dilation)


@traceable
def blockwise_dropout_conv2d(input, kernel, block_size, p: float, padding=(0, 0), stride=(1, 1),
                             dilation=(1, 1), seed: int | None = None) -> torch.Tensor:
    """Block-dropout convolution with a fresh mask over the patch matrix, drawn on the device by a launch that
    the call needs anyway (``seed`` pins it, as for the matmul; gather and product of a pinned draw each evaluate it)."""
    if not 0 <= p < 1:
        raise ValueError("Dropout probability must be in [0, 1)")
    bs = _block_size(block_size)
    if bs % 64:
        raise NotImplementedError(f"block_size {bs}: the convolution takes multiples of 64 (the matmul also 32)")
    return _conv2d(input, kernel, None, bs, p, padding, stride, dilation, draw_source(input, seed))


def naive_blockwise_dropout_conv2d_mask(input, mask, block_size, p: float, kernel, padding=(0, 0),
                                        stride=(1, 1), dilation=(1, 1)) -> torch.Tensor:
    """The same function in plain torch ops (unfold, expanded mask, dense linear); no work skipped."""
    from .naive import blockwise_dropout_matmul_mask

    n, c, h, w = input.shape
    k, _, r, s = kernel.shape
    po, qo = GEMM.conv_out_hw(h, w, r, s, _pair(padding), _pair(stride), _pair(dilation))
    cols = F.unfold(input, (r, s), dilation=_pair(dilation), padding=_pair(padding), stride=_pair(stride))
    cols = cols.permute(0, 2, 1).reshape(n * po * qo, c * r * s)
    y2 = blockwise_dropout_matmul_mask(cols, mask, block_size, p, kernel.reshape(k, -1))
    return y2.view(n, po * qo, k).permute(0, 2, 1).reshape(n, k, po, qo)


def naive_blockwise_dropout_conv2d(input, kernel, block_size, p: float, padding=(0, 0), stride=(1, 1),
                                   dilation=(1, 1)) -> torch.Tensor:
    bs = _block_size(block_size)
    rows, ncols = conv_patch_matrix_shape(input.shape, kernel.shape, padding, stride, dilation)
    mask = torch.rand(ceil(rows / bs), ceil(ncols / bs), device=input.device) < p
    return naive_blockwise_dropout_conv2d_mask(input, mask, bs, p, kernel, padding, stride, dilation)
