"""Layers whose widths are not multiples of 8 or whose operands start off 16-byte boundaries: their products run on
copies with padded rows, and must be what the oracle says, over contiguous results of the true sizes."""
import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, cpu_mask, make_operand, max_tile_rel_fro, rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu


def _check(x, w, dy, bs, p, gen):
    import flash_dropout.functional as F

    (M, K), N = x.shape, w.shape[0]
    mask = cpu_mask(O.mask_shape(M, K, bs), p, gen)
    mk = mask.numpy()
    x.requires_grad_()
    w.requires_grad_()
    y = F.hip_blockwise_dropout_matmul_mask(x, mask.cuda(), bs, p, w)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    assert y.is_contiguous() and dx.is_contiguous() and dw.is_contiguous()
    xn, wn, dyn = to_np(x), to_np(w), to_np(dy)
    for got, ref, what in ((y, O.dsd_forward(xn, wn, mk, bs, p, np.float32), "y"),
                           (dx, O.sdd_dx(dyn, wn, mk, bs, p, np.float32), "dx"),
                           (dw, O.dsd_dw(dyn, xn, mk, bs, p, np.float32), "dw")):
        assert max_tile_rel_fro(got, ref) <= REL_FRO_TOL, what  # fp32 sums, rounded once: orders of magnitude of room
    assert (dx.float().cpu().numpy()[~O.expand_keep(mk, bs, M, K)] == 0).all()


@pytest.mark.parametrize("M,N,K,bs,p", [
    (1, 1, 1, 64, 0.0),           # one element
    (63, 7, 65, 64, 0.3),         # one past a block, a row shorter than one 16-byte piece
    (130, 64, 127, 32, 0.5),      # only the reduction is odd, quadrant keep bits
    (200, 129, 128, 64, 0.4),     # only the output is odd
    (257, 515, 1025, 96, 0.3),
    (2100, 1031, 333, 128, 0.2),  # 128 x 128 tiles
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_any_width(M, N, K, bs, p, dtype):
    gen = torch.Generator().manual_seed(M + 5 * N + K)
    x = make_operand(M, K, dtype, "cuda", gen=gen)
    w = make_operand(N, K, dtype, "cuda", scale=K ** -0.5, gen=gen)
    _check(x, w, make_operand(M, N, dtype, "cuda", gen=gen), bs, p, gen)


def test_operands_off_their_boundaries():
    """Slices that start 2 bytes behind a boundary (last rows end where their storage ends), a column-major gradient."""
    gen = torch.Generator().manual_seed(3)
    wide = make_operand(150, 137, torch.float16, "cuda", gen=gen)
    ws = make_operand(80, 137, torch.float16, "cuda", gen=gen)
    for dy in (make_operand(150, 81, torch.float16, "cuda", gen=gen)[:, 1:],
               make_operand(150, 80, torch.float16, "cuda", row_major=False, gen=gen)):
        _check(wide[:, 1:].detach(), ws[:, 1:].detach(), dy, 64, 0.4, gen)


@pytest.mark.parametrize("dims", [(33, 64, 10), (72, 65, 31, 3)])
@pytest.mark.parametrize("act", ["relu", "gelu"])
def test_stack_of_odd_widths(dims, act):
    """A stack whose first layer runs dense (no dropout, no input gradient) against the oracle with hidden tensors rounded
    to fp16 where the kernels round them.  An unrounded reference has other ReLU masks: of some 3000 hidden values of
    spread 0.4, one or two lie within a rounding (2^-11 relative on 65 terms) of zero, and each one that crosses moves a
    weight gradient by one of about 1500 equal outer products, 1 / sqrt(1500) = 2.6 % of its norm."""
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(sum(dims))
    x = torch.rand(100, dims[0], generator=gen).half().cuda()
    ws = [make_operand(o, i, torch.float16, "cuda", scale=i ** -0.5, gen=gen).requires_grad_() for i, o in zip(dims, dims[1:])]
    dy = make_operand(100, dims[-1], torch.float16, "cuda", gen=gen)
    y = F.hip_blockwise_dropout_mlp(x, ws, 64, 0.0, act)
    got = torch.autograd.grad(y, ws, dy)
    keep = [np.zeros(O.mask_shape(100, i, 64), dtype=bool) for i in dims[:-1]]
    out, _, dws = O.mlp_forward_backward(to_np(x), [to_np(w) for w in ws], keep, 64, 0.0, act, to_np(dy), hidden_dtype=np.float16)
    for a, b in zip((y, *got), (out, *dws)):
        assert rel_fro(a, b) <= REL_FRO_TOL
