"""Kernel (e): im2col gather / col2im and the conv path built on them, against the CPU oracle."""
import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, max_tile_rel_fro, cpu_mask, rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu

GEOMS = [
    dict(n=2, c=3, h=8, w=8, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),
    dict(n=3, c=5, h=13, w=9, r=3, s=2, padding=(0, 1), stride=(2, 1), dilation=(1, 2)),
    dict(n=4, c=64, h=16, w=16, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),
    dict(n=2, c=16, h=10, w=10, r=1, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)),
    dict(n=1, c=8, h=12, w=12, r=5, s=5, padding=(2, 2), stride=(2, 2), dilation=(1, 1)),
    # P*Q a multiple of 64 and C*R*S a multiple of 8: the patch-staged im2col kernel
    dict(n=2, c=24, h=24, w=24, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),   # 216 columns: ragged tile
    dict(n=2, c=8, h=32, w=32, r=3, s=3, padding=(1, 1), stride=(2, 2), dilation=(1, 1)),
    dict(n=1, c=16, h=16, w=16, r=3, s=3, padding=(2, 2), stride=(1, 1), dilation=(2, 2)),
    dict(n=2, c=8, h=16, w=16, r=5, s=5, padding=(2, 2), stride=(1, 1), dilation=(1, 1)),
    dict(n=1, c=32, h=8, w=128, r=1, s=7, padding=(0, 3), stride=(1, 1), dilation=(1, 1)),   # a 64-row group inside one image row
]


def _geo(cfg):
    return dict(padding=cfg["padding"], stride=cfg["stride"], dilation=cfg["dilation"])


@pytest.mark.parametrize("cfg", GEOMS)
@pytest.mark.parametrize("channels_last", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_im2col_bit_exact(cfg, channels_last, dtype):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(0)
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).to(dtype)
    xg = x.cuda()
    if channels_last:
        xg = xg.contiguous(memory_format=torch.channels_last)
    cols = GEMM().im2col(xg, (cfg["r"], cfg["s"]), **_geo(cfg))
    ref = O.im2col(x.float().numpy(), cfg["r"], cfg["s"], **_geo(cfg))
    assert cols.shape == ref.shape
    assert np.array_equal(cols.float().cpu().numpy(), ref)  # a gather: bit exact


@pytest.mark.parametrize("cfg", [
    GEOMS[2],                                                                                   # patch-staged kernel
    dict(n=4, c=64, h=12, w=12, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),      # P*Q = 144: tile-turning kernel
    dict(n=4, c=24, h=16, w=16, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),      # 216 columns: ragged last block
])
@pytest.mark.parametrize("bs", [64, 128])
def test_im2col_writes_only_kept_blocks(cfg, bs):
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(1)
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half().cuda()
    ks = (cfg["r"], cfg["s"])
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], *ks, **_geo(cfg))
    rows, ncols = cfg["n"] * p_ * q_, cfg["c"] * cfg["r"] * cfg["s"]
    mask = cpu_mask(O.mask_shape(rows, ncols, bs), 0.5, gen)
    lists = ext.build_lists(mask.cuda())
    full = ext.im2col(x, ks, **_geo(cfg))
    part = torch.full((rows, ncols), 7.0, dtype=torch.float16, device="cuda")
    ext.im2col(x, ks, lists=lists, block_size=bs, out=part, **_geo(cfg))
    keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, rows, ncols)).cuda()
    assert torch.equal(part[keep], full[keep])
    assert bool((part[~keep] == 7.0).all())  # dropped blocks are not touched


@pytest.mark.parametrize("cfg", [
    dict(n=1, c=40, h=8, w=8, r=5, s=5, padding=(2, 2), stride=(1, 1), dilation=(1, 1)),     # 1 row group, 16 column tiles: one to a workgroup
    dict(n=3, c=208, h=8, w=8, r=5, s=5, padding=(2, 2), stride=(2, 2), dilation=(1, 1)),    # 82 tiles, the last ragged
    dict(n=7, c=232, h=7, w=7, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),    # 6 row groups, 33 tiles
    dict(n=20, c=96, h=24, w=24, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),  # 180 row groups: some tiles to a workgroup
])
@pytest.mark.parametrize("channels_last", [False, True])
@pytest.mark.parametrize("p,bs", [(None, 64), (0.5, 64), (0.9, 64), (0.5, 128), (0.5, 192)])
def test_im2col_of_few_rows_deals_out_its_columns(cfg, channels_last, p, bs):
    """Few row groups: the column tiles, or the kept ones of them, are dealt out over workgroups.  A gather, so bit exact, with
    every kept block written and no other."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(cfg["c"])
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half()
    ks = (cfg["r"], cfg["s"])
    ref = torch.from_numpy(O.im2col(x.float().numpy(), *ks, **_geo(cfg))).half()
    xg = x.cuda()
    if channels_last:
        xg = xg.contiguous(memory_format=torch.channels_last)
    if p is None:
        assert torch.equal(ext.im2col(xg, ks, **_geo(cfg)).cpu(), ref)
        return
    mask = cpu_mask(O.mask_shape(*ref.shape, bs), p, gen)
    lists = ext.build_lists(mask.cuda())
    part = torch.full(ref.shape, 7.0, dtype=torch.float16, device="cuda")
    ext.im2col(xg, ks, lists=lists, block_size=bs, out=part, **_geo(cfg))
    keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, *ref.shape))
    assert torch.equal(part.cpu(), torch.where(keep, ref, torch.tensor(7.0, dtype=torch.float16)))


@pytest.mark.parametrize("c,h,w,padding,r,s", [
    (16, 12, 24, (1, 1), 3, 3),    # rows in pieces of 8 pixels
    (16, 6, 28, (2, 2), 5, 5),     # of 4
    (24, 7, 14, (0, 3), 2, 7),     # of 2, more padding than a piece
    (8, 9, 15, (1, 1), 3, 3),      # one by one
    (40, 8, 8, (9, 9), 3, 3),      # padding past a row's length
    (72, 10, 10, (0, 0), 1, 1),    # channels last: pieces of 8 channels, tiles that start inside one
    (8, 20, 48, (1, 1), 5, 5),     # 2.56 channels to a tile
    (12, 11, 13, (1, 1), 3, 3),    # channels one by one
])
@pytest.mark.parametrize("stride", [(1, 1), (2, 2), (2, 1)])
@pytest.mark.parametrize("layout", ["planes", "channels_last", "cropped", "channels", "offset"])
def test_im2col_copies_in_pieces(c, h, w, padding, r, s, stride, layout):
    """Images whose rows or pixels can be copied several elements at a time, and slices of larger ones that cannot."""
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(w)
    n, geo = 3, dict(padding=padding, stride=stride, dilation=(1, 1))
    if layout == "cropped":      # rows four pixels longer than the image's
        x = torch.randn(n, c, h, w + 4, generator=gen).half().cuda()[..., 2:2 + w]
    elif layout == "channels":   # some of a channels-last image's channels
        x = torch.randn(n, c + 5, h, w, generator=gen).half().cuda().contiguous(memory_format=torch.channels_last)[:, 3:3 + c]
    elif layout == "offset":     # a tensor that starts 2 bytes behind a boundary
        x = torch.randn(n * c * h * w + 1, generator=gen).half().cuda()[1:].view(n, c, h, w)
    else:
        x = torch.randn(n, c, h, w, generator=gen).half().cuda()
        if layout == "channels_last":
            x = x.contiguous(memory_format=torch.channels_last)
    cols = GEMM().im2col(x, (r, s), **geo)
    ref = O.im2col(x.float().cpu().numpy(), r, s, **geo)
    assert np.array_equal(cols.float().cpu().numpy(), ref)


@pytest.mark.parametrize("cfg", GEOMS)
@pytest.mark.parametrize("channels_last", [False, True])
def test_col2im_vs_oracle(cfg, channels_last):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(2)
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    rows, ncols = cfg["n"] * p_ * q_, cfg["c"] * cfg["r"] * cfg["s"]
    g = torch.randn(rows, ncols, generator=gen).half()
    shape = (cfg["n"], cfg["c"], cfg["h"], cfg["w"])
    dx = GEMM().col2im(g.cuda(), shape, (cfg["r"], cfg["s"]), channels_last=channels_last, **_geo(cfg))
    ref = O.col2im(g.float().numpy(), shape, cfg["r"], cfg["s"], **_geo(cfg))
    assert dx.shape == shape
    assert rel_fro(dx, ref) <= 2e-3  # fp32 sum of <= R*S fp16 values, one rounding
    # with a mask: dropped blocks count as zero and are not read
    mask = cpu_mask(O.mask_shape(rows, ncols, 64), 0.5, gen)
    keep = O.expand_keep(mask.numpy(), 64, rows, ncols)
    dxm = GEMM().col2im(g.cuda(), shape, (cfg["r"], cfg["s"]), mask=mask.cuda(), block_size=64, **_geo(cfg))
    refm = O.col2im(np.where(keep, g.float().numpy(), 0), shape, cfg["r"], cfg["s"], **_geo(cfg))
    assert rel_fro(dxm, refm) <= 2e-3


@pytest.mark.parametrize("cfg", [
    dict(n=2, c=16, h=48, w=48, r=3, s=3, padding=(1, 1)),   # 24 x 24 outputs: the last row and column of the image meet one tap
    dict(n=2, c=8, h=7, w=9, r=3, s=3, padding=(1, 1)),      # odd sizes
    dict(n=2, c=24, h=14, w=14, r=1, s=1, padding=(0, 0)),   # three pixels in four meet no tap: zeros
    dict(n=2, c=8, h=14, w=13, r=1, s=1, padding=(1, 1)),
    dict(n=2, c=16, h=33, w=20, r=5, s=5, padding=(2, 2)),
    dict(n=1, c=8, h=17, w=11, r=5, s=5, padding=(0, 3)),    # no padding down: the first and the last rows meet fewer taps
    dict(n=2, c=8, h=12, w=16, r=2, s=2, padding=(0, 0)),    # taps by loop counters
    dict(n=1, c=8, h=13, w=10, r=4, s=3, padding=(3, 1)),
    dict(n=1, c=8, h=9, w=200, r=7, s=3, padding=(3, 1)),    # rows so long that the band shrinks
    dict(n=3, c=8, h=10, w=10, r=3, s=3, padding=(2, 2)),    # more padding than the kernel reaches over
])
@pytest.mark.parametrize("channels_last", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [None, 64, 128])
def test_col2im_with_stride_two(cfg, channels_last, dtype, bs):
    from flash_dropout.hip import GEMM

    geo = dict(padding=cfg["padding"], stride=(2, 2), dilation=(1, 1))
    gen = torch.Generator().manual_seed(cfg["h"])
    shape, ks = (cfg["n"], cfg["c"], cfg["h"], cfg["w"]), (cfg["r"], cfg["s"])
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], *ks, **geo)
    rows, ncols = cfg["n"] * p_ * q_, cfg["c"] * cfg["r"] * cfg["s"]
    g = torch.randn(rows, ncols, generator=gen).to(dtype)
    given, mask = g.clone(), None
    if bs:
        mask = cpu_mask(O.mask_shape(rows, ncols, bs), 0.4, gen)
        keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, rows, ncols))
        given[~keep] = float("nan")  # dropped blocks are not read
        g = torch.where(keep, g, torch.zeros_like(g))
        mask = mask.cuda()
    dx = GEMM().col2im(given.cuda(), shape, ks, mask=mask, block_size=bs, channels_last=channels_last, **geo)
    ref = torch.from_numpy(O.col2im(g.double().numpy(), shape, *ks, **geo))
    # one rounding to the element type of a sum of fewer than 32 terms in fp32
    eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert bool(((dx.cpu().double() - ref).abs() <= eps * ref.abs() + 2.0 ** -18).all())


# pixels and channels that fill a tile of 64 and that do not, images that start and end inside a block of rows
@pytest.mark.parametrize("n,c,h,w", [(3, 64, 8, 8), (2, 8, 7, 7), (5, 72, 9, 15), (1, 130, 3, 70), (4, 65, 1, 5), (3, 1, 16, 12), (2, 200, 20, 13)])
@pytest.mark.parametrize("bs", [None, 64, 128, 192])
@pytest.mark.parametrize("sliced", [False, True])
def test_col2im_of_pointwise_kernels(n, c, h, w, bs, sliced):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(n * c + h)
    rows = n * h * w
    g = torch.randn(rows, c, generator=gen).half()
    given, mask = g.clone(), None
    if bs:
        mask = cpu_mask(O.mask_shape(rows, c, bs), 0.4, gen)
        keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, rows, c))
        given[~keep] = float("nan")  # dropped blocks are not read
        g = torch.where(keep, g, torch.zeros_like(g))
        mask = mask.cuda()
    given = given.cuda()
    if sliced:  # rows that start on any boundary
        given = torch.cat([given.new_zeros(rows, 3), given], 1)[:, 3:]
    dx = GEMM().col2im(given, (n, c, h, w), (1, 1), mask=mask, block_size=bs)
    assert torch.equal(dx.cpu(), g.reshape(n, h * w, c).permute(0, 2, 1).reshape(n, c, h, w))


@pytest.mark.parametrize("n,c,h,w,k", [(9, 72, 15, 13, 40), (3, 24, 56, 56, 72), (20, 104, 7, 7, 100), (2, 200, 30, 30, 64)])
@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("sliced", [False, True])
def test_pointwise_convolutions_of_planes_and_of_pixels_agree(n, c, h, w, k, bs, sliced):
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(c)
    x = torch.randn(n, c + 8 * sliced, h, w, generator=gen).half().cuda()[:, 4 * sliced:][:, :c]
    wt = (torch.randn(k, c, 1, 1, generator=gen) * c ** -0.5).half().cuda().requires_grad_()
    dy = torch.randn(n, k, h, w, generator=gen).half().cuda()
    got = []
    for image in (x, x.contiguous(memory_format=torch.channels_last)):
        image = image.detach().requires_grad_()
        y = F.blockwise_dropout_conv2d(image, wt, bs, 0.4, 0, 1, seed=11)
        got.append((y, *torch.autograd.grad(y, (image, wt), dy)))
    assert all(torch.equal(a, b) for a, b in zip(*got))


# two, three and four groups of channels to a workgroup, the last with fewer, in one band and in two of unequal height
@pytest.mark.parametrize("cfg", [
    dict(n=600, c=56, h=6, w=5, r=3, padding=(1, 1), stride=(2, 2)),
    dict(n=850, c=64, h=4, w=7, r=3, padding=(1, 1), stride=(1, 1)),
    dict(n=700, c=48, h=11, w=6, r=3, padding=(0, 2), stride=(2, 2)),
    dict(n=300, c=120, h=9, w=4, r=5, padding=(2, 2), stride=(2, 2)),
    dict(n=280, c=64, h=9, w=19, r=5, padding=(2, 2), stride=(2, 2)),  # windows of more than 30 KB: 512 threads
    dict(n=520, c=64, h=6, w=7, r=5, padding=(2, 1), stride=(1, 1)),
])
@pytest.mark.parametrize("bs,p", [(None, 0.0), (64, 0.5), (192, 0.3)])
@pytest.mark.parametrize("channels_last", [False, True])
def test_col2im_of_many_workgroups(cfg, bs, p, channels_last):
    from flash_dropout.hip import GEMM

    geo = dict(padding=cfg["padding"], stride=cfg["stride"], dilation=(1, 1))
    shape, ks = (cfg["n"], cfg["c"], cfg["h"], cfg["w"]), (cfg["r"], cfg["r"])
    assert cfg["n"] * (cfg["c"] // 8) * -(-cfg["h"] // 8) >= 4096
    gen = torch.Generator().manual_seed(cfg["n"])
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], *ks, **geo)
    rows, ncols = cfg["n"] * p_ * q_, cfg["c"] * cfg["r"] ** 2
    g = torch.randn(rows, ncols, generator=gen).half()
    given, mask = g.clone(), None
    if bs:
        mask = cpu_mask(O.mask_shape(rows, ncols, bs), p, gen)
        keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, rows, ncols))
        given[~keep] = float("nan")  # dropped blocks are not read
        g = torch.where(keep, g, torch.zeros_like(g))
        mask = mask.cuda()
    dx = GEMM().col2im(given.cuda(), shape, ks, mask=mask, block_size=bs, channels_last=channels_last, **geo)
    ref = torch.nn.functional.fold(g.double().reshape(cfg["n"], p_ * q_, ncols).permute(0, 2, 1), shape[2:], ks, padding=cfg["padding"],
                                   stride=cfg["stride"])
    assert bool(((dx.cpu().double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 2.0 ** -18).all())  # as above


@pytest.mark.parametrize("cfg", [
    dict(n=8, c=64, h=32, w=32, k=128, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),
    dict(n=4, c=24, h=17, w=15, k=40, r=3, s=3, padding=(1, 0), stride=(2, 1), dilation=(1, 1)),
])
@pytest.mark.parametrize("p", [0.0, 0.5])
def test_blockdrop_conv_forward_backward(cfg, p):
    """Reduced-batch version of the conv configuration (same 64->128 3x3 stride 1 pad 1 layer, 8 images
    instead of 128) plus a ragged geometry: forward, dx and dkernel against the oracle."""
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(5)
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half()
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    k = ((torch.rand(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * 2 - 1) * fan_in ** -0.5).half()
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    rows = cfg["n"] * p_ * q_
    mask = cpu_mask(O.mask_shape(rows, fan_in, 64), p, gen)
    dy = torch.randn(cfg["n"], cfg["k"], p_, q_, generator=gen).half()

    xg, kg = x.cuda().requires_grad_(), k.cuda().requires_grad_()
    y = F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), 64, p, kg, **_geo(cfg))
    assert y.shape == dy.shape
    y.backward(dy.cuda())
    ry, rdx, rdk = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), 64, p, dy=to_np(dy), dtype=np.float32, **_geo(cfg))
    assert max_tile_rel_fro(y, ry) <= REL_FRO_TOL
    assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
    assert max_tile_rel_fro(kg.grad, rdk) <= REL_FRO_TOL


IMPLICIT_GEOMS = [
    # (geometry, taken by the implicit kernel)
    (dict(n=4, c=64, h=32, w=32, k=128, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),   # the conv configuration's layer
    (dict(n=2, c=16, h=16, w=16, k=40, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),    # 144 columns, 40 outputs: ragged both ways; 4 output rows per block
    (dict(n=3, c=8, h=32, w=32, k=64, r=5, s=5, padding=(2, 2), stride=(1, 1), dilation=(1, 1)), True),     # 25 taps
    (dict(n=2, c=64, h=32, w=32, k=256, r=1, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),   # 1x1: one reduction block, two column tiles
    (dict(n=2, c=32, h=16, w=64, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),    # one output row per block
    (dict(n=5, c=24, h=32, w=8, k=72, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),     # 8 output rows per block
    (dict(n=2, c=16, h=36, w=32, k=64, r=5, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),    # no padding: P = 32 from H = 36
    (dict(n=2, c=16, h=16, w=16, k=64, r=3, s=3, padding=(2, 2), stride=(1, 1), dilation=(1, 1)), False),   # Q = 18
    (dict(n=2, c=8, h=32, w=32, k=64, r=3, s=3, padding=(1, 1), stride=(2, 2), dilation=(1, 1)), True),     # stride 2: 16 x 16 outputs
    (dict(n=2, c=24, h=32, w=32, k=64, r=3, s=3, padding=(2, 2), stride=(1, 1), dilation=(2, 2)), True),    # dilation 2
    (dict(n=3, c=16, h=32, w=32, k=72, r=3, s=3, padding=(1, 1), stride=(2, 1), dilation=(1, 1)), True),    # stride 2 down, 1 across
    (dict(n=2, c=40, h=64, w=16, k=64, r=5, s=3, padding=(4, 1), stride=(2, 2), dilation=(2, 1)), True),    # stride and dilation, Q = 8
    (dict(n=1, c=16, h=8, w=16, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),     # P*Q = 128: every 64-position block with its own input rows, half a workgroup
    (dict(n=5, c=32, h=8, w=8, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),      # 8 x 8 images: a workgroup's four blocks are four images, the last workgroup has one
    (dict(n=3, c=72, h=12, w=16, k=136, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),   # P*Q = 192: blocks of 4 rows, three per image, 648 columns
    (dict(n=1, c=256, h=32, w=32, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),   # too many channels for one copy of the input rows: a copy per step
    (dict(n=2, c=136, h=16, w=16, k=192, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),  # the same with 1224 columns (ragged), two column tiles
]


@pytest.fixture(params=["auto", "big"])
def copy_form(request):
    """The implicit forward keeps a copy of the input rows per step, or one copy of all channels' rows for the
    whole kernel where only that fits; the large-tile policy prefers the latter, so both run where both fit."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    prev = ext.set_tile_policy(request.param)
    yield request.param
    ext.set_tile_policy(prev)


@pytest.mark.parametrize("cfg,taken", IMPLICIT_GEOMS)
@pytest.mark.parametrize("p", [0.0, 0.5])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_implicit_gemm_conv_forward(cfg, taken, p, dtype, copy_form):
    """sd_conv2d_dsd_lists (no patch matrix) against the oracle and against im2col + DSD on the same lists;
    geometries it does not take must come back as None with nothing written."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(cfg["c"] + cfg["k"])
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).to(dtype)
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    k = ((torch.rand(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * 2 - 1) * fan_in ** -0.5).to(dtype)
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    rows = cfg["n"] * p_ * q_
    mask = cpu_mask(O.mask_shape(rows, fan_in, 64), p, gen)
    lists = ext.build_lists(mask.cuda())
    xg, w2 = x.cuda(), k.cuda().reshape(cfg["k"], fan_in)
    s = 1 / (1 - p)
    y = ext.conv2d_dsd_lists(xg, w2, lists, 64, s, (cfg["r"], cfg["s"]), **_geo(cfg))
    if not taken:
        assert y is None
        return
    assert y is not None and tuple(y.shape) == (rows, cfg["k"])
    assert ext.last_kernel() == "specialised"
    cols = ext.im2col(xg, (cfg["r"], cfg["s"]), **_geo(cfg))
    explicit = ext.gemm_dsd_lists(cols, w2, lists, 64, s)
    assert rel_fro(y, to_np(explicit)) <= 1e-3
    ry = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), 64, p, dtype=np.float32, **_geo(cfg))
    ry2 = np.transpose(ry, (0, 2, 3, 1)).reshape(rows, cfg["k"])
    assert max_tile_rel_fro(y, ry2) <= REL_FRO_TOL


@pytest.mark.parametrize("cfg,taken", [g for g in IMPLICIT_GEOMS if g[1]][:5] + IMPLICIT_GEOMS[-2:])
def test_implicit_gemm_conv_dense(cfg, taken, copy_form):
    """No lists = every block kept: the dense convolution, against torch's conv2d in fp32."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(2)
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half()
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    k = ((torch.rand(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * 2 - 1) * fan_in ** -0.5).half()
    y = ext.conv2d_dsd_lists(x.cuda(), k.cuda().reshape(cfg["k"], fan_in), None, 0, 1.0, (cfg["r"], cfg["s"]), **_geo(cfg))
    assert y is not None
    ref = torch.nn.functional.conv2d(x.float(), k.float(), padding=cfg["padding"])
    n, kk, p_, q_ = ref.shape
    assert max_tile_rel_fro(y, ref.permute(0, 2, 3, 1).reshape(n * p_ * q_, kk).numpy()) <= REL_FRO_TOL


@pytest.mark.parametrize("cfg,fwd_taken", IMPLICIT_GEOMS)
@pytest.mark.parametrize("p", [0.0, 0.5])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_implicit_gemm_conv_weight_gradient(cfg, fwd_taken, p, dtype):
    """sd_conv2d_dw_lists (no patch matrix) against the oracle and against im2col + DSD on the transposed
    operands; it takes every geometry the forward takes (and some more: P*Q only has to be a multiple of 64)."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(cfg["c"] * 3 + cfg["k"])
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).to(dtype)
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    rows = cfg["n"] * p_ * q_
    dy2 = torch.randn(rows, cfg["k"], generator=gen).to(dtype)
    mask = cpu_mask(O.mask_shape(rows, fan_in, 64), p, gen)
    lists = ext.build_lists(mask.cuda())
    s = 1 / (1 - p)
    xg, dyg = x.cuda(), dy2.cuda()
    dw = ext.conv2d_dw_lists(xg, dyg, lists, 64, s, (cfg["r"], cfg["s"]), **_geo(cfg))
    if dw is None:
        assert not fwd_taken
        return
    assert tuple(dw.shape) == (cfg["k"], fan_in)
    cols = ext.im2col(xg, (cfg["r"], cfg["s"]), **_geo(cfg))
    explicit = ext.gemm_dsd_lists(cols.t(), dyg.t(), lists.transposed(), 64, s, transposed_out=True).t()
    assert rel_fro(dw, to_np(explicit)) <= 2e-3
    ref = O.dsd_dw(to_np(dy2), O.im2col(to_np(x), cfg["r"], cfg["s"], **_geo(cfg)), mask.numpy(), 64, p, np.float32)
    assert max_tile_rel_fro(dw, ref) <= REL_FRO_TOL
    if p == 0.0:  # and without lists: the dense weight gradient
        dense = ext.conv2d_dw_lists(xg, dyg, None, 0, 1.0, (cfg["r"], cfg["s"]), **_geo(cfg))
        assert dense is not None and max_tile_rel_fro(dense, ref) <= REL_FRO_TOL


DX_GEOMS = [
    (dict(n=4, c=64, h=32, w=32, k=128, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),   # the conv configuration's layer
    (dict(n=2, c=16, h=16, w=16, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),    # 144 columns: ragged last block
    (dict(n=2, c=16, h=33, w=33, k=128, r=2, s=2, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),   # 2x2 on a 33 x 33 image: one block column, 18 open channels
    (dict(n=2, c=64, h=32, w=32, k=128, r=1, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),   # 1x1: 66 open channels per block column, so the band shrinks to one input row for the ring to fit
    (dict(n=2, c=32, h=16, w=64, k=64, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),    # one output row per block
    (dict(n=3, c=24, h=32, w=8, k=128, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),    # 8 output rows per block
    (dict(n=2, c=16, h=34, w=32, k=64, r=3, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),    # no padding, H not a multiple of the band
    (dict(n=2, c=8, h=16, w=16, k=64, r=5, s=5, padding=(2, 2), stride=(1, 1), dilation=(1, 1)), True),     # 25 taps, 4 output rows per block
    (dict(n=2, c=128, h=16, w=16, k=256, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), True),  # K_out = 256: the instance with the longer reduction
    (dict(n=2, c=24, h=16, w=16, k=192, r=5, s=3, padding=(2, 1), stride=(1, 1), dilation=(1, 1)), True),   # K_out = 192, 15 taps
    (dict(n=2, c=16, h=32, w=32, k=256, r=1, s=1, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), True),   # 1x1 with K_out = 256: that instance's LDS holds the 66-slot ring
    (dict(n=1, c=16, h=32, w=32, k=320, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), False),  # K_out = 320
    (dict(n=2, c=40, h=32, w=32, k=128, r=2, s=2, padding=(0, 0), stride=(1, 1), dilation=(1, 1)), False),  # Q = 31
    (dict(n=3, c=8, h=32, w=32, k=64, r=5, s=5, padding=(2, 2), stride=(1, 1), dilation=(1, 1)), True),     # 5 taps high on 2-row blocks: the band shrinks to two input rows
    (dict(n=2, c=16, h=16, w=16, k=40, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)), False),   # K_out = 40
    (dict(n=2, c=8, h=32, w=32, k=64, r=3, s=3, padding=(1, 1), stride=(2, 2), dilation=(1, 1)), True),     # stride 2: three of four taps fall between outputs
    (dict(n=2, c=24, h=32, w=32, k=64, r=3, s=3, padding=(2, 2), stride=(1, 1), dilation=(2, 2)), True),    # dilation 2
    (dict(n=3, c=16, h=32, w=32, k=128, r=3, s=3, padding=(1, 1), stride=(2, 1), dilation=(1, 1)), True),   # stride 2 down, 1 across
    (dict(n=2, c=40, h=64, w=16, k=64, r=5, s=3, padding=(4, 1), stride=(2, 2), dilation=(2, 1)), True),    # stride and dilation, Q = 8
]


@pytest.mark.parametrize("cfg,taken", DX_GEOMS)
@pytest.mark.parametrize("p", [0.0, 0.5])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("channels_last", [False, True])
def test_fused_conv_input_gradient(cfg, taken, p, dtype, channels_last):
    """sd_conv2d_dx (kept tiles of dY.W formed and folded in LDS) against the oracle's dx and against the
    two-kernel route; run twice, the result must be bitwise the same (one owner and one order per sum)."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(cfg["c"] * 5 + cfg["k"])
    shape = (cfg["n"], cfg["c"], cfg["h"], cfg["w"])
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    kern = ((torch.rand(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * 2 - 1) * fan_in ** -0.5).to(dtype)
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    rows = cfg["n"] * p_ * q_
    dy2 = torch.randn(rows, cfg["k"], generator=gen).to(dtype)
    mask = cpu_mask(O.mask_shape(rows, fan_in, 64), p, gen)
    s = 1 / (1 - p)
    w2 = kern.cuda().reshape(cfg["k"], fan_in)
    dx = ext.conv2d_dx(dy2.cuda(), w2, shape, (cfg["r"], cfg["s"]), mask=mask.cuda(), block_size=64, scale=s,
                       channels_last=channels_last, **_geo(cfg))
    if not taken:
        assert dx is None
        return
    assert dx is not None and tuple(dx.shape) == shape
    again = ext.conv2d_dx(dy2.cuda(), w2, shape, (cfg["r"], cfg["s"]), mask=mask.cuda(), block_size=64, scale=s,
                          channels_last=channels_last, **_geo(cfg))
    assert torch.equal(dx, again)
    lists = ext.build_lists(mask.cuda())
    dcols = ext.gemm_sdd_lists(dy2.cuda(), w2.t(), lists, 64, s)
    two_step = ext.col2im(dcols, shape, (cfg["r"], cfg["s"]), mask=mask.cuda(), block_size=64, **_geo(cfg))
    assert rel_fro(dx, to_np(two_step)) <= 2e-3
    ref = O.col2im(O.sdd_dx(to_np(dy2), to_np(w2.cpu()), mask.numpy(), 64, p, np.float32), shape, cfg["r"], cfg["s"],
                   **_geo(cfg))
    assert max_tile_rel_fro(dx, ref) <= REL_FRO_TOL
    if p == 0.0:  # no mask: the dense input gradient
        dense = ext.conv2d_dx(dy2.cuda(), w2, shape, (cfg["r"], cfg["s"]), **_geo(cfg))
        assert dense is not None and max_tile_rel_fro(dense, ref) <= REL_FRO_TOL


@pytest.mark.parametrize("stride,dilation,padding", [((1, 1), (1, 1), (1, 1)), ((2, 2), (1, 1), (1, 1)),
                                                     ((1, 1), (2, 2), (2, 2))])
def test_implicit_and_explicit_conv_routes_agree(stride, dilation, padding):
    """The autograd function with the implicit forward (input kept, kept patch blocks re-gathered for the weight
    gradient, fused input gradient) and with the explicit one (patch matrix kept) give the same three results,
    also for a strided and for a dilated convolution."""
    import sys

    import flash_dropout.functional as F

    mod = sys.modules["flash_dropout.functional.im2col_conv2d"]  # the package re-exports a function of that name
    gen = torch.Generator().manual_seed(9)
    x = torch.randn(4, 64, 32, 32, generator=gen).half().cuda()
    k = (torch.randn(128, 64, 3, 3, generator=gen) * 0.04).half().cuda()
    p_, q_ = O.conv_out_hw(32, 32, 3, 3, padding=padding, stride=stride, dilation=dilation)
    dy = torch.randn(4, 128, p_, q_, generator=gen).half().cuda()
    mask = (torch.rand(4 * p_ * q_ // 64, 9, generator=gen) < 0.5).cuda()
    out = {}
    for implicit in (True, False):
        prev, mod.IMPLICIT_FORWARD = mod.IMPLICIT_FORWARD, implicit
        prev_dx, mod.FUSED_INPUT_GRADIENT = mod.FUSED_INPUT_GRADIENT, implicit
        try:
            xg, kg = x.clone().requires_grad_(), k.clone().requires_grad_()
            y = F.blockwise_dropout_conv2d_mask(xg, mask, 64, 0.5, kg, padding=padding, stride=stride,
                                                dilation=dilation)
            y.backward(dy)
            out[implicit] = (y.detach(), xg.grad, kg.grad)
        finally:
            mod.IMPLICIT_FORWARD = prev
            mod.FUSED_INPUT_GRADIENT = prev_dx
    for a, b, what in zip(out[True], out[False], ("y", "dx", "dk")):
        assert rel_fro(a, to_np(b)) <= 1e-3, what


@pytest.mark.parametrize("dropout", [True, False])
def test_conv_backward_takes_an_expanded_gradient(dropout):
    """out.sum().backward() hands the backward a gradient with all strides zero; it must be laid out before the
    kernels see it (the result is then the gradient of the sum: compare with a materialised gradient of ones)."""
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(3)
    x = torch.randn(4, 16, 16, 16, generator=gen).half().cuda()
    k = (torch.randn(64, 16, 3, 3, generator=gen) * 0.08).half().cuda()
    mask = (torch.rand(16, 3, generator=gen) < 0.5).cuda()
    grads = []
    for expanded in (True, False):
        xg, kg = x.clone().requires_grad_(), k.clone().requires_grad_()
        if dropout:
            out = F.blockwise_dropout_conv2d_mask(xg, mask, 64, 0.5, kg, padding=(1, 1))
        else:
            out = F.im2col_conv2d(xg, kg, padding=(1, 1), stride=(1, 1), dilation=(1, 1))
        if expanded:
            out.sum().backward()
        else:
            out.backward(torch.ones_like(out))
        grads.append((xg.grad, kg.grad))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
    assert grads[0][0].abs().sum().item() > 0


def test_dense_im2col_conv_matches_conv2d():
    """The reference's implied check for its im2col path: equal to F.conv2d (benchmark/conv.py:20-75)."""
    import flash_dropout.functional as F

    torch.manual_seed(6)
    x = torch.randn(4, 32, 20, 20, device="cuda", dtype=torch.float16, requires_grad=True)
    k = (torch.randn(48, 32, 3, 3, device="cuda", dtype=torch.float16) * 0.06).requires_grad_()
    y = F.im2col_conv2d(x, k, padding=(1, 1), stride=(1, 1), dilation=(1, 1))
    dy = torch.randn_like(y)
    y.backward(dy)
    xr, kr = x.detach().float().requires_grad_(), k.detach().float().requires_grad_()
    yr = torch.nn.functional.conv2d(xr, kr, padding=1)
    yr.backward(dy.float())
    assert max_tile_rel_fro(y, yr) <= REL_FRO_TOL
    assert max_tile_rel_fro(x.grad, xr.grad) <= REL_FRO_TOL
    assert max_tile_rel_fro(k.grad, kr.grad) <= REL_FRO_TOL


def test_conv_layer_variants_on_gpu():
    from flash_dropout.layers import DropoutConv2d

    torch.manual_seed(7)
    x = torch.randn(4, 16, 12, 12, device="cuda", dtype=torch.float16)
    for variant in ("im2col", "blockwise[hip]", "blockwise[naive]"):
        conv = DropoutConv2d(16, 32, (3, 3), padding=(1, 1), p=0.0, variant=variant, block_size=64).cuda().half()
        ref = torch.nn.functional.conv2d(x, conv.weight, padding=1)
        assert max_tile_rel_fro(conv(x), ref) <= REL_FRO_TOL, variant
    conv = DropoutConv2d(16, 32, (3, 3), padding=(1, 1), p=0.5, variant="blockwise[hip]", block_size=64).cuda().half()
    y = conv(x)
    y.float().sum().backward()
    assert y.shape == (4, 32, 12, 12) and conv.weight.grad is not None


def test_full_size_conv_config_against_the_full_oracle():
    """The full conv configuration ([128,64,32,32] -> patch matrix [131072 x 576], 3x3 64->128, p = 0.5) at full
    batch: forward, input gradient and weight gradient (2048 row blocks, the reduction split over workgroups)
    against the fp32 oracle, every tile; plus the adjoint identity <im2col(x), g> == <x, col2im(g)>."""
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(8)
    geo = dict(padding=(1, 1), stride=(1, 1), dilation=(1, 1))
    x = torch.randn(128, 64, 32, 32, generator=gen).half()
    k = ((torch.rand(128, 64, 3, 3, generator=gen) * 2 - 1) * 576 ** -0.5).half()
    mask = cpu_mask((2048, 9), 0.5, gen)
    dy = torch.randn(128, 128, 32, 32, generator=gen).half()
    xg, kg = x.cuda().requires_grad_(), k.cuda().requires_grad_()
    y = F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), 64, 0.5, kg, **geo)
    y.backward(dy.cuda())
    # none of the three products went through a patch matrix
    assert F.conv_last_routes() == {"forward": "implicit", "dx": "fused", "dw": "implicit"}
    ry, rdx, rdk = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), 64, 0.5, dy=to_np(dy), dtype=np.float32, **geo)
    # in the products' own layouts, so that a tile of the check is a tile of the kernels
    as_rows = lambda t: t.permute(0, 2, 3, 1).reshape(-1, t.shape[1])
    assert max_tile_rel_fro(as_rows(y.detach().cpu()), as_rows(torch.from_numpy(ry))) <= REL_FRO_TOL
    assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
    assert max_tile_rel_fro(kg.grad.reshape(128, 576), rdk.reshape(128, 576)) <= REL_FRO_TOL
    xs = x[:16].cuda()
    cols = ext.im2col(xs, (3, 3), **geo)
    g = torch.randn(cols.shape, generator=gen).half().cuda()
    lhs = (cols.double() * g.double()).sum().item()
    rhs = (xs.double() * ext.col2im(g, xs.shape, (3, 3), **geo).double()).sum().item()
    assert abs(lhs - rhs) <= 2e-3 * max(abs(lhs), (cols.double().norm() * g.double().norm()).item() * 1e-2)


@pytest.mark.parametrize("bs,dx_route", [(64, "fused"), (128, "fused"), (192, "fused")])
def test_conv_routes_are_reported_and_block_sizes_above_64_stay_fused(bs, dx_route):
    """Which route a convolution's products took is visible (conv_last_routes), a geometry the fused kernels do not take
    reports the patch-matrix route, and masks at block sizes 128 and 192 run the fused input gradient too (as the
    mask of the same elements at block size 64): results against the oracle at that block size."""
    import sys

    import flash_dropout.functional as F

    mod = sys.modules["flash_dropout.functional.im2col_conv2d"]  # the package re-exports a function of that name

    gen = torch.Generator().manual_seed(12)
    geo = dict(padding=(1, 1), stride=(1, 1), dilation=(1, 1))
    x = torch.randn(8, 64, 32, 32, generator=gen).half()
    k = ((torch.rand(128, 64, 3, 3, generator=gen) * 2 - 1) * 576 ** -0.5).half()
    dy = torch.randn(8, 128, 32, 32, generator=gen).half()
    mask = cpu_mask(O.mask_shape(8 * 32 * 32, 576, bs), 0.5, gen)
    xg, kg = x.cuda().requires_grad_(), k.cuda().requires_grad_()
    y = F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), bs, 0.5, kg, **geo)
    y.backward(dy.cuda())
    assert F.conv_last_routes() == {"forward": "implicit", "dx": dx_route, "dw": "implicit"}
    ry, rdx, rdk = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), bs, 0.5, dy=to_np(dy), dtype=np.float32, **geo)
    assert max_tile_rel_fro(y, ry) <= REL_FRO_TOL
    assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
    assert max_tile_rel_fro(kg.grad, rdk) <= REL_FRO_TOL
    if bs == 64:
        # Q = 18 is a geometry none of the fused kernels takes; and the switches force the patch-matrix route
        x2 = torch.randn(2, 16, 16, 16, generator=gen).half().cuda().requires_grad_()
        k2 = (torch.randn(64, 16, 3, 3, generator=gen) * 144 ** -0.5).half().cuda().requires_grad_()
        F.im2col_conv2d(x2, k2, padding=(2, 2)).sum().backward()
        assert F.conv_last_routes() == {"forward": "explicit", "dx": "explicit", "dw": "explicit"}
        old = mod.IMPLICIT_FORWARD, mod.FUSED_INPUT_GRADIENT
        try:
            mod.IMPLICIT_FORWARD = mod.FUSED_INPUT_GRADIENT = False
            xg.grad = kg.grad = None
            F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), bs, 0.5, kg, **geo).backward(dy.cuda())
            assert F.conv_last_routes() == {"forward": "explicit", "dx": "explicit", "dw": "explicit"}
            assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
        finally:
            mod.IMPLICIT_FORWARD, mod.FUSED_INPUT_GRADIENT = old


@pytest.mark.parametrize("cfg,p,routes", [
    # few rows: gather and small tiles
    (dict(n=9, c=24, h=8, w=8, k=64, r=3, s=3, stride=(1, 1), padding=(1, 1)), 0.5, ("explicit", "explicit", "explicit")),
    (dict(n=6, c=16, h=16, w=16, k=64, r=5, s=5, stride=(2, 2), padding=(2, 2)), 0.3, ("explicit", "explicit", "explicit")),
    (dict(n=4, c=16, h=32, w=32, k=64, r=2, s=2, stride=(2, 2), padding=(0, 0)), 0.0, ("explicit", "fused", "explicit")),  # one block wide
    # 63 and 64 workgroups of the implicit forward, below 8192 rows and not
    (dict(n=31, c=8, h=32, w=32, k=64, r=3, s=3, stride=(2, 2), padding=(1, 1)), 0.3, ("explicit", "explicit", "explicit")),
    (dict(n=63, c=8, h=32, w=32, k=64, r=3, s=3, stride=(2, 2), padding=(1, 1)), 0.3, ("explicit", "explicit", "implicit")),
    (dict(n=64, c=8, h=32, w=32, k=64, r=3, s=3, stride=(2, 2), padding=(1, 1)), 0.3, ("implicit", "explicit", "implicit")),
    # pointwise kernels: planes of up to 64 MB are turned, by two the forward stays implicit, the kernel's gradient from 16384 rows on
    (dict(n=15, c=16, h=32, w=32, k=64, r=1, s=1, stride=(1, 1), padding=(0, 0)), 0.3, ("explicit", "fused", "explicit")),
    (dict(n=16, c=16, h=32, w=32, k=64, r=1, s=1, stride=(1, 1), padding=(0, 0)), 0.3, ("explicit", "fused", "explicit")),
    (dict(n=15, c=16, h=64, w=64, k=64, r=1, s=1, stride=(2, 2), padding=(0, 0)), 0.3, ("implicit", "explicit", "explicit")),
    (dict(n=16, c=16, h=64, w=64, k=64, r=1, s=1, stride=(2, 2), padding=(0, 0)), 0.3, ("implicit", "explicit", "implicit")),
    (dict(n=128, c=64, h=64, w=64, k=64, r=1, s=1, stride=(1, 1), padding=(0, 0)), 0.3, ("explicit", "explicit", "explicit")),  # 64 MB
    (dict(n=129, c=64, h=64, w=64, k=64, r=1, s=1, stride=(1, 1), padding=(0, 0)), 0.3, ("implicit", "explicit", "implicit")),
    # 300 MB of patch gradient stay out of memory
    (dict(n=192, c=32, h=64, w=64, k=64, r=5, s=5, stride=(2, 2), padding=(2, 2)), 0.9, ("implicit", "fused", "implicit")),
])
def test_masked_convolutions_go_through_a_patch_matrix_where_that_is_faster(cfg, p, routes):
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(cfg["n"])
    geo = dict(padding=cfg["padding"], stride=cfg["stride"], dilation=(1, 1))
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half()
    k = (torch.randn(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * fan_in ** -0.5).half()
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **geo)
    rows = cfg["n"] * p_ * q_
    mask = cpu_mask(O.mask_shape(rows, fan_in, 64), p, gen)
    dy = torch.randn(cfg["n"], cfg["k"], p_, q_, generator=gen).half()
    xg, kg = x.cuda().requires_grad_(), k.cuda().requires_grad_()
    call = lambda: F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), 64, p, kg, **geo)
    y = call()
    y.backward(dy.cuda())
    assert tuple(F.conv_last_routes()[n] for n in ("forward", "dx", "dw")) == routes
    if cfg["n"] < 100:
        ry, rdx, rdk = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), 64, p, dy=to_np(dy), dtype=np.float32, **geo)
        assert max_tile_rel_fro(y, ry) <= REL_FRO_TOL
        assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
        assert max_tile_rel_fro(kg.grad, rdk) <= REL_FRO_TOL
    # the image is kept, whichever way the products went: a write to it before the backward is refused
    y = call()
    with torch.no_grad():
        xg.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy.cuda())
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
        y = call()
    assert tuple(x.shape) in kept and (rows, fan_in) not in kept
    y.backward(dy.cuda())


@pytest.mark.parametrize("cfg", [
    dict(n=3, c=208, h=8, w=8, r=5, s=5, padding=(2, 2), stride=(2, 2), dilation=(1, 1)),    # 82 tiles over workgroups, the last ragged
    dict(n=20, c=24, h=14, w=14, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),  # ragged rows
    dict(n=1, c=5, h=9, w=260, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),    # rows off 16-byte boundaries: the turning kernel
])
@pytest.mark.parametrize("bs", [64, 128, 192])
@pytest.mark.parametrize("source", ["given", "given by columns", "seed"])
def test_im2col_of_a_mask_source_writes_the_blocks_of_its_lists(cfg, bs, source):
    """The gather that asks the mask itself against the bytes that the list builder stores of the same draw."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(bs)
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half().cuda()
    ks = (cfg["r"], cfg["s"])
    ref = torch.from_numpy(O.im2col(x.float().cpu().numpy(), *ks, **_geo(cfg))).half()
    shape = O.mask_shape(*ref.shape, bs)
    mask, seed = None, 0
    if source.startswith("given"):
        mask = cpu_mask(shape, 0.4, gen).cuda()
        if "columns" in source:
            mask = mask.t().contiguous().t()
    else:
        seed = 91
    part = torch.full(ref.shape, 7.0, dtype=torch.float16, device="cuda")
    rc = ext.lib.sd_im2col_masked(x.data_ptr(), *x.stride(), part.data_ptr(), part.stride(0), *x.shape, *ks, *cfg["padding"],
                                  *cfg["stride"], *cfg["dilation"], None if mask is None else mask.data_ptr(),
                                  *((0, 0) if mask is None else mask.stride()), seed, 0, 0.4, bs, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    if mask is None:
        mask = ext.random_lists(shape, 0.4, seed=seed, device=x.device)[0]
    keep = torch.from_numpy(O.expand_keep(mask.cpu().numpy(), bs, *ref.shape))
    assert torch.equal(part.cpu(), torch.where(keep, ref, torch.tensor(7.0, dtype=torch.float16)))


@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("c,k,r,stride", [(16, 40, 3, 1), (24, 72, 5, 2), (72, 64, 1, 2)])
@pytest.mark.parametrize("channels_last", [False, True])
def test_both_gradients_through_the_patch_matrix_match_one_at_a_time(bs, c, k, r, stride, channels_last):
    """One launch for both products, dropped blocks of the patch gradient left as they are, against one product at a time."""
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(c)
    x = torch.randn(7, c, 14, 14, generator=gen).half().cuda()
    if channels_last:
        x = x.contiguous(memory_format=torch.channels_last)
    w = (torch.randn(k, c, r, r, generator=gen) * (c * r * r) ** -0.5).half().cuda().requires_grad_()
    x.requires_grad_()
    y = F.blockwise_dropout_conv2d(x, w, bs, 0.4, r // 2, stride, seed=3)
    dy = torch.randn(y.shape, generator=gen).half().cuda()
    both = torch.autograd.grad(y, (x, w), dy, retain_graph=True)
    assert F.conv_last_routes()["dx"] == "explicit" and both[0].stride() == x.stride()
    for one, wrt in zip(both, (x, w)):
        alone, = torch.autograd.grad(y, wrt, dy, retain_graph=True)
        # sums in fp32 in another order, one rounding to fp16 of a product and, for dx, one of the fold
        assert rel_fro(one, to_np(alone)) <= 1e-3


@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("c,k,r,stride", [(16, 40, 3, 1), (72, 64, 1, 2), (24, 64, 5, 2)])
def test_conv_draws_of_the_generator_state_are_those_of_its_seed(bs, c, k, r, stride):
    """A draw of the state is made by one launch and read from what it stored, one of a seed by gather and product each: the same
    mask, results equal to rounding, and the state moves on by one draw a call."""
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(c)
    x = torch.randn(7, c, 14, 14, generator=gen).half().cuda().requires_grad_()
    w = (torch.randn(k, c, r, r, generator=gen) * (c * r * r) ** -0.5).half().cuda().requires_grad_()
    ext.manual_seed(77)
    try:
        y = F.blockwise_dropout_conv2d(x, w, bs, 0.4, r // 2, stride)
        assert ext.rng_state(x.device).tolist() == [77, 1, 0, 0]
        pinned = F.blockwise_dropout_conv2d(x, w, bs, 0.4, r // 2, stride, seed=77)
        dy = torch.randn(y.shape, generator=gen).half().cuda()
        grads, pinned_grads = (torch.autograd.grad(v, (x, w), dy) for v in (y, pinned))
        # sums in fp32 in another order at most, one rounding to fp16 of a product and, for dx, one of the fold
        for one, other in zip((y, *grads), (pinned, *pinned_grads)):
            assert rel_fro(one, to_np(other)) <= 1e-3
    finally:
        ext.manual_seed(torch.initial_seed())


# folds that run one thread to an element: channels that do not fill groups of eight, windows by two that do not fit the LDS
@pytest.mark.parametrize("cfg", [
    dict(n=3, c=12, h=13, w=9, r=3, s=3, padding=(1, 1), stride=(1, 1), dilation=(1, 1)),
    dict(n=5, c=5, h=10, w=11, r=4, s=2, padding=(2, 0), stride=(2, 3), dilation=(1, 2)),
    dict(n=2, c=8, h=7, w=300, r=3, s=3, padding=(1, 1), stride=(2, 2), dilation=(1, 1)),
    dict(n=2, c=8, h=33, w=32, r=7, s=7, padding=(3, 3), stride=(2, 2), dilation=(1, 1)),
    dict(n=1, c=16, h=100, w=96, r=5, s=5, padding=(2, 2), stride=(2, 2), dilation=(1, 1)),
])
# 65535: a block size whose reciprocal is exact for no image at all
@pytest.mark.parametrize("bs", [1, 30, 64, 72, 96, 192, 65535])
@pytest.mark.parametrize("by_columns", [False, True])
def test_masked_folds_of_single_elements(cfg, bs, by_columns):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(cfg["w"] + bs)
    shape, ks = (cfg["n"], cfg["c"], cfg["h"], cfg["w"]), (cfg["r"], cfg["s"])
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], *ks, **_geo(cfg))
    rows, ncols = cfg["n"] * p_ * q_, cfg["c"] * cfg["r"] * cfg["s"]
    g = torch.randn(rows, ncols, generator=gen).half()
    mask = torch.rand(O.mask_shape(rows, ncols, bs), generator=gen) < 0.4
    keep = torch.from_numpy(O.expand_keep(mask.numpy(), bs, rows, ncols))
    given = torch.where(keep, g, torch.tensor(float("nan"), dtype=g.dtype))  # dropped blocks are not read
    mask = mask.cuda()
    if by_columns:
        mask = mask.t().contiguous().t()
    dx = GEMM().col2im(given.cuda(), shape, ks, mask=mask, block_size=bs, **_geo(cfg))
    kept = torch.where(keep, g, torch.zeros_like(g)).double()
    ref, size = (torch.from_numpy(O.col2im(t.numpy(), shape, *ks, **_geo(cfg))) for t in (kept, kept.abs()))
    # one rounding to fp16 of a sum of fewer than 64 terms in fp32
    assert bool(((dx.cpu().double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 2.0 ** -18 * size + 2.0 ** -25).all())


@pytest.mark.parametrize("cfg,dx", [
    # folds that the tile kernel would do stay with the fused input gradient
    (dict(n=6, c=32, h=32, w=32, k=64, r=3, s=3, stride=(2, 1), padding=(1, 1), dilation=(1, 1)), "fused"),
    (dict(n=6, c=32, h=32, w=32, k=64, r=3, s=3, stride=(1, 2), padding=(1, 1), dilation=(1, 1)), "fused"),
    (dict(n=5, c=32, h=32, w=32, k=64, r=3, s=3, stride=(2, 2), padding=(2, 2), dilation=(2, 2)), "fused"),
    (dict(n=4, c=8, h=32, w=64, k=128, r=4, s=4, stride=(4, 4), padding=(0, 0), dilation=(1, 1)), "fused"),
    # and long folds of single elements at unit strides, where there are few outputs
    (dict(n=100, c=10, h=17, w=33, k=64, r=4, s=4, stride=(1, 1), padding=(1, 1), dilation=(1, 1)), "fused"),
    (dict(n=60, c=10, h=17, w=33, k=64, r=4, s=4, stride=(1, 1), padding=(1, 1), dilation=(1, 1)), "explicit"),
    (dict(n=100, c=10, h=17, w=33, k=128, r=4, s=4, stride=(1, 1), padding=(1, 1), dilation=(1, 1)), "explicit"),
    # by windows, element by element
    (dict(n=6, c=32, h=32, w=32, k=64, r=3, s=3, stride=(2, 2), padding=(1, 1), dilation=(1, 1)), "explicit"),
    (dict(n=6, c=12, h=32, w=32, k=64, r=4, s=4, stride=(2, 2), padding=(1, 1), dilation=(1, 1)), "explicit"),
    (dict(n=3, c=16, h=32, w=32, k=64, r=7, s=7, stride=(2, 2), padding=(3, 3), dilation=(1, 1)), "explicit"),
])
@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("channels_last", [False, True])
def test_the_fused_input_gradient_is_replaced_where_the_fold_is_fast(cfg, dx, bs, channels_last):
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(cfg["r"])
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half()
    k = (torch.randn(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * fan_in ** -0.5).half()
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    mask = cpu_mask(O.mask_shape(cfg["n"] * p_ * q_, fan_in, bs), 0.4, gen)
    dy = torch.randn(cfg["n"], cfg["k"], p_, q_, generator=gen).half()
    xg, kg = x.cuda(), k.cuda().requires_grad_()
    if channels_last:
        xg = xg.contiguous(memory_format=torch.channels_last)
    xg.requires_grad_()
    y = F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), bs, 0.4, kg, **_geo(cfg))
    y.backward(dy.cuda())
    assert F.conv_last_routes()["dx"] == dx
    ry, rdx, rdk = O.conv2d_blockdrop(to_np(x), to_np(k), mask.numpy(), bs, 0.4, dy=to_np(dy), dtype=np.float32, **_geo(cfg))
    assert max_tile_rel_fro(y, ry) <= REL_FRO_TOL
    assert max_tile_rel_fro(xg.grad, rdx) <= REL_FRO_TOL
    assert max_tile_rel_fro(kg.grad, rdk) <= REL_FRO_TOL


@pytest.mark.parametrize("bs", [64, 128, 192])
@pytest.mark.parametrize("n,c,h,w,k", [(7, 72, 14, 14, 64), (1, 8, 3, 2, 8), (9, 200, 15, 13, 40), (20, 20, 16, 16, 24)])
def test_pointwise_draws_of_the_generator_state_are_those_of_its_seed(bs, n, c, h, w, k):
    """The launch that turns the planes draws the mask (for widths that are no multiple of 8 the lists' launch does): the same lists,
    so the same bits, and the state moves on by one draw a call, captured ones too."""
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(c)
    x = torch.randn(n, c, h, w, generator=gen).half().cuda().requires_grad_()
    wt = (torch.randn(k, c, 1, 1, generator=gen) * c ** -0.5).half().cuda().requires_grad_()
    dy = torch.randn(n, k, h, w, generator=gen).half().cuda()
    passed = lambda y: (y, *torch.autograd.grad(y, (x, wt), dy))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    try:
        with torch.cuda.stream(stream):
            ext.manual_seed(77)
            drawn = passed(F.blockwise_dropout_conv2d(x, wt, bs, 0.4))
            assert F.conv_last_routes()["forward"] == "explicit"
            assert ext.rng_state(x.device).tolist() == [77, 1, 0, 0]
            pinned = passed(F.blockwise_dropout_conv2d(x, wt, bs, 0.4, seed=77))
            if c % 8 == 0:
                assert all(torch.equal(a, b) for a, b in zip(drawn, pinned))
            else:  # sums in fp32 in another order, one rounding to fp16 of a product and, for dx, one of the fold
                assert all(rel_fro(a, to_np(b)) <= 1e-3 for a, b in zip(drawn, pinned))
            y = F.blockwise_dropout_conv2d(x.detach(), wt, bs, 0.4, seed=77)
            assert rel_fro(torch.autograd.grad(y, wt, dy)[0], to_np(pinned[2])) <= 1e-3  # on its own, as above
            with torch.no_grad():
                want = [F.blockwise_dropout_conv2d(x, wt, bs, 0.4) for _ in range(3)]
                ext.manual_seed(77)
                F.blockwise_dropout_conv2d(x, wt, bs, 0.4)
                stream.synchronize()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=stream):
                    y = F.blockwise_dropout_conv2d(x, wt, bs, 0.4)
                for draw in want:
                    graph.replay()
                    assert torch.equal(y, draw)
    finally:
        torch.cuda.synchronize()
        ext.manual_seed(torch.initial_seed())


@pytest.mark.parametrize("cfg", [
    dict(n=32, c=24, h=32, w=32, k=128, r=3, s=3, stride=(2, 1), padding=(1, 1), dilation=(1, 1)),
    dict(n=64, c=24, h=32, w=32, k=128, r=3, s=3, stride=(2, 2), padding=(2, 2), dilation=(2, 2)),
    dict(n=64, c=16, h=32, w=32, k=128, r=2, s=2, stride=(2, 2), padding=(0, 0), dilation=(1, 1)),  # one block column
])
def test_strided_convolutions_without_and_with_a_patch_matrix_agree(cfg):
    """Layers whose three products need no patch matrix, off the tap-wise route, against the same with the switches off."""
    import sys

    import flash_dropout.functional as F

    mod = sys.modules["flash_dropout.functional.im2col_conv2d"]  # the package re-exports a function of that name
    gen = torch.Generator().manual_seed(cfg["n"])
    fan_in = cfg["c"] * cfg["r"] * cfg["s"]
    x = torch.randn(cfg["n"], cfg["c"], cfg["h"], cfg["w"], generator=gen).half().cuda()
    k = (torch.randn(cfg["k"], cfg["c"], cfg["r"], cfg["s"], generator=gen) * fan_in ** -0.5).half().cuda()
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], cfg["r"], cfg["s"], **_geo(cfg))
    dy = torch.randn(cfg["n"], cfg["k"], p_, q_, generator=gen).half().cuda()
    mask = cpu_mask(O.mask_shape(cfg["n"] * p_ * q_, fan_in, 64), 0.5, gen).cuda()
    out = []
    for routes in (("implicit", "fused", "implicit"), ("explicit", "explicit", "explicit")):
        old = mod.IMPLICIT_FORWARD, mod.FUSED_INPUT_GRADIENT
        mod.IMPLICIT_FORWARD = mod.FUSED_INPUT_GRADIENT = routes[0] == "implicit"
        try:
            xg, kg = x.clone().requires_grad_(), k.clone().requires_grad_()
            y = F.blockwise_dropout_conv2d_mask(xg, mask, 64, 0.5, kg, **_geo(cfg))
            y.backward(dy)
            assert tuple(F.conv_last_routes()[name] for name in ("forward", "dx", "dw")) == routes
            out.append((y.detach(), xg.grad, kg.grad))
        finally:
            mod.IMPLICIT_FORWARD, mod.FUSED_INPUT_GRADIENT = old
    for a, b, what in zip(*out, ("y", "dx", "dk")):
        # sums in fp32 in another order, one rounding to fp16 of a product and, for dx, one of the fold
        assert rel_fro(a, to_np(b)) <= 1e-3, what


# masks of blocks larger than the kernel's 64: rows and columns that end inside a block of the mask
@pytest.mark.parametrize("cfg", [
    dict(n=3, c=24, h=8, w=8, k=64, r=3, s=3, stride=(1, 1), padding=(1, 1), dilation=(1, 1)),      # 192 rows, 216 columns
    dict(n=5, c=40, h=32, w=32, k=128, r=3, s=3, stride=(2, 2), padding=(1, 1), dilation=(1, 1)),   # 1280 rows, 360 columns
    dict(n=1, c=16, h=16, w=16, k=192, r=5, s=3, stride=(2, 1), padding=(2, 1), dilation=(1, 1)),   # one image, 128 rows
])
@pytest.mark.parametrize("bs", [64, 128, 192, 1024])
@pytest.mark.parametrize("by_columns", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_input_gradient_reads_masks_of_larger_blocks(cfg, bs, by_columns, dtype):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(cfg["c"] + bs)
    shape, ks = (cfg["n"], cfg["c"], cfg["h"], cfg["w"]), (cfg["r"], cfg["s"])
    cols = cfg["c"] * cfg["r"] * cfg["s"]
    p_, q_ = O.conv_out_hw(cfg["h"], cfg["w"], *ks, **_geo(cfg))
    rows = cfg["n"] * p_ * q_
    dy2 = torch.randn(rows, cfg["k"], generator=gen).to(dtype).cuda()
    w2 = (torch.randn(cfg["k"], cols, generator=gen) * cfg["k"] ** -0.5).to(dtype).cuda()
    mask = cpu_mask(O.mask_shape(rows, cols, bs), 0.4, gen)
    given = mask.t().contiguous().t().cuda() if by_columns else mask.cuda()
    strides = (1, max(given.shape[0], 1)) if by_columns else (given.shape[1], 1)
    dx = torch.full(shape, float("nan"), dtype=dtype, device="cuda")
    rc = GEMM().lib.sd_conv2d_dx_blocks(dy2.data_ptr(), dy2.stride(0), w2.data_ptr(), w2.stride(0), dx.data_ptr(), *dx.stride(),
                                        given.data_ptr(), *strides, *shape, cfg["k"], *ks, *cfg["padding"], *cfg["stride"],
                                        *cfg["dilation"], bs, 1 / 0.6, int(dtype == torch.bfloat16),
                                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    ref = O.col2im(O.sdd_dx(to_np(dy2), to_np(w2), mask.numpy(), bs, 0.4, np.float32), shape, *ks, **_geo(cfg))
    assert max_tile_rel_fro(dx, ref) <= REL_FRO_TOL
    # the same mask in blocks of 64: the same bits
    fine = mask.repeat_interleave(bs // 64, 0).repeat_interleave(bs // 64, 1)[:-(-rows // 64), :-(-cols // 64)].contiguous().cuda()
    assert torch.equal(dx, GEMM().conv2d_dx(dy2, w2, shape, ks, mask=fine, block_size=64, scale=1 / 0.6, **_geo(cfg)))


@pytest.mark.parametrize("c,hw,r,stride", [(24, 16, 1, 1), (9, 7, 1, 1), (16, 32, 3, 2), (24, 8, 5, 1), (32, 28, 3, 1)])
@pytest.mark.parametrize("channels_last", [False, True])
def test_every_route_refuses_kernels_without_outputs_and_rates_that_round_to_one(c, hw, r, stride, channels_last):
    import flash_dropout.functional as F

    x = torch.ones(6, c, hw, hw, device="cuda", dtype=torch.float16)
    if channels_last:
        x = x.contiguous(memory_format=torch.channels_last)
    wt = torch.ones(40, c, r, r, device="cuda", dtype=torch.float16)
    for seed in (3, None):
        with pytest.raises(ValueError):
            F.blockwise_dropout_conv2d(x, wt[:0], 64, 0.4, r // 2, stride, seed=seed)
        with pytest.raises(ValueError):
            F.blockwise_dropout_conv2d(x, wt, 64, 1 - 1e-9, r // 2, stride, seed=seed)
    with pytest.raises(ValueError):
        F.im2col_conv2d(x, wt[:0], r // 2, stride)
