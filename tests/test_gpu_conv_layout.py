"""The convolution's data movement at its edges: 64-row groups that end inside an image or span several, column groups
that need more than one copy of the input rows, and the gradient's planes turned into rows."""
import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, cpu_mask, max_tile_rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,hw,r,stride,pad,dil", [
    (3, 8, 28, 3, 1, 1, 1),     # 784 positions: groups across two images, the last one ragged
    (9, 16, 7, 3, 1, 1, 1),     # 49 positions: up to three images to a group
    (70, 8, 3, 3, 2, 1, 1),     # 4 positions an image: 16 or 17 images to a group
    (2, 8, 30, 5, 2, 2, 1),     # stride 2, 225 positions
    (2, 8, 33, 3, 1, 2, 2),     # dilation, rows longer than half a wave
    (2, 200, 14, 3, 1, 1, 1),   # more channels than one copy holds
    (5, 24, 9, 1, 1, 0, 1),     # 1 x 1
])
@pytest.mark.parametrize("bs", [64, 128])
def test_patch_matrix_any_image_size(n, c, hw, r, stride, pad, dil, bs):
    """Bit exact (a gather), whole and kept blocks only; nothing outside the kept blocks is written."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    geo = dict(padding=(pad, pad), stride=(stride, stride), dilation=(dil, dil))
    gen = torch.Generator().manual_seed(n * c + hw)
    x = torch.randn(n, c, hw, hw, generator=gen).half()
    ref = O.im2col(x.float().numpy(), r, r, **geo)
    full = ext.im2col(x.cuda(), (r, r), **geo)
    assert np.array_equal(full.float().cpu().numpy(), ref)
    mask = cpu_mask(O.mask_shape(*ref.shape, bs), 0.5, gen)
    part = torch.full_like(full, 7.0)
    ext.im2col(x.cuda(), (r, r), lists=ext.build_lists(mask.cuda()), block_size=bs, out=part, **geo)
    keep = O.expand_keep(mask.numpy(), bs, *ref.shape)
    assert np.array_equal(part.float().cpu().numpy(), np.where(keep, ref, 7.0))


@pytest.mark.parametrize("n,c,p", [(1, 2, 2), (2, 64, 64), (3, 65, 63), (2, 130, 784), (5, 7, 49), (1, 128, 1)])
@pytest.mark.parametrize("gap", [0, 3])
def test_rows_from_planes(n, c, p, gap):
    """Bit exact at the edges of the 64 x 64 tiles; planes `gap` elements apart start on any 2-byte boundary."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    store = torch.randint(-30000, 30000, (n, c, p + gap), dtype=torch.int16, device="cuda")
    src = store[:, :, gap:]
    dst = torch.full((n * p + 1, c), 77, dtype=torch.int16, device="cuda")
    ext._call(ext.lib.sd_rows_from_planes, src.data_ptr(), src.stride(0), src.stride(1), dst.data_ptr(), n, c, p, ext._stream(dst))
    assert torch.equal(dst[:-1].view(n, p, c), src.transpose(1, 2)) and (dst[-1] == 77).all()


@pytest.mark.parametrize("n,c,hw,k", [(3, 40, 9, 24), (2, 96, 14, 168), (1, 8, 3, 8)])
@pytest.mark.parametrize("p", [0.0, 0.5])
def test_pointwise_convolution_of_pixel_rows(n, c, hw, k, p):
    """1 x 1 on a channels-last image: its pixels are the patch matrix and the patch gradient, dropped blocks zero."""
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(c)
    x = torch.randn(n, c, hw, hw, generator=gen).half().cuda().to(memory_format=torch.channels_last).requires_grad_()
    w = (torch.randn(k, c, 1, 1, generator=gen) * c ** -0.5).half().cuda().requires_grad_()
    mask = cpu_mask(O.mask_shape(n * hw * hw, c, 64), p, gen)
    y = F.blockwise_dropout_conv2d_mask(x, mask.cuda(), 64, p, w)
    dy = torch.randn(*y.shape, generator=gen).half().cuda()
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    assert dx.shape == x.shape and dx.is_contiguous(memory_format=torch.channels_last)
    rows = lambda t: to_np(t.permute(0, 2, 3, 1).reshape(n * hw * hw, -1))
    xn, wn, dyn = rows(x), to_np(w).reshape(k, c), rows(dy)
    for got, ref in ((rows(y), O.dsd_forward(xn, wn, mask.numpy(), 64, p, np.float32)),
                     (rows(dx), O.sdd_dx(dyn, wn, mask.numpy(), 64, p, np.float32)),
                     (to_np(dw).reshape(k, c), O.dsd_dw(dyn, xn, mask.numpy(), 64, p, np.float32))):
        assert max_tile_rel_fro(got, ref) <= REL_FRO_TOL
