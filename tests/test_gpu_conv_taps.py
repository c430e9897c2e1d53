"""The tap-wise convolution (csrc/conv_taps.hip): all three products against the oracle at the sizes where its windows, tiles
and masks end."""
import ctypes as C

import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, cpu_mask, max_tile_rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu

# n, c, h, w, k, r, s, padding, dilation: images that end inside a 16-position tile, windows over several images and over the
# first and last row, a channel tile more or less than a step, tap groups of nine with a rest, results larger and
# smaller than the image
GEOMS = [
    (5, 32, 7, 7, 40, 3, 3, (1, 1), (1, 1)),
    (3, 40, 14, 14, 136, 3, 3, (1, 1), (1, 1)),
    (2, 72, 28, 28, 32, 3, 3, (1, 1), (1, 1)),
    (2, 136, 16, 16, 200, 3, 3, (1, 1), (1, 1)),
    (2, 64, 30, 30, 64, 5, 5, (2, 2), (1, 1)),
    (3, 8, 9, 64, 72, 3, 3, (1, 1), (1, 1)),
    (4, 48, 12, 10, 8, 3, 2, (0, 1), (1, 2)),
    (4, 32, 6, 9, 64, 3, 3, (3, 4), (1, 1)),
    (2, 24, 20, 18, 96, 3, 3, (2, 2), (2, 2)),
    (9, 64, 3, 3, 64, 3, 3, (1, 1), (1, 1)),
    (2, 32, 1, 40, 64, 1, 7, (0, 3), (1, 1)),
    (1, 16, 3, 3, 16, 2, 2, (0, 0), (1, 1)),  # four output positions
    # gradients narrower than the image: the planes of dX are turned in more LDS than its products use
    (40, 64, 8, 11, 64, 1, 9, (0, 0), (1, 1)),
    (30, 72, 5, 11, 40, 1, 3, (0, 0), (1, 4)),
    (20, 40, 6, 15, 72, 1, 12, (0, 0), (1, 1)),
    # windows of 784, 912 and 992 rows (1000 are the most): the weight gradient has LDS for one buffer of them
    (1, 32, 9, 256, 40, 3, 3, (1, 1), (1, 1)),
    (1, 40, 8, 160, 64, 5, 5, (2, 2), (1, 1)),
    (1, 24, 7, 360, 72, 3, 3, (1, 1), (1, 1)),
]


def _tensors(geom, dtype, seed=0):
    n, c, h, w, k, r, s, pad, dil = geom
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(n, c, h, w, generator=gen).to(dtype)
    wt = (torch.randn(k, c, r, s, generator=gen) * (c * r * s) ** -0.5).to(dtype)
    po, qo = O.conv_out_hw(h, w, r, s, padding=pad, stride=(1, 1), dilation=dil)
    return x, wt, torch.randn(n, k, po, qo, generator=gen).to(dtype), n * po * qo, gen


def _products(geom, x, wt, dy, mask, bs, scale, channels_last=False):
    """y, dx, dw through the library's entry points, whatever route a layer of this size would take."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    lib, call = ext.lib, ext._call
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy = x.cuda(), wt.cuda(), dy.cuda()
    dt = 1 if x.dtype == torch.bfloat16 else 0
    geo = (n, c, h, w, k, r, s, *pad, 1, 1, *dil)
    assert lib.sd_conv2d_taps_fits(*geo) == 1
    pixels = dy.shape[2] * dy.shape[3]
    rows = n * pixels
    new = lambda *shape: torch.empty(*shape, dtype=x.dtype, device="cuda")
    array = lambda t, *v: (t * len(v))(*v)
    xr, dyr, y, dw = new(n * h * w, c), new(rows, k), new(rows, k), new(k, c * r * s)
    packed = [new(lib.sd_conv2d_taps_packed_bytes(c, k, r, s, b) // 2) for b in (0, 1)]
    st = ext._stream(x)
    for b, (src, dst, ch, px) in enumerate(((x, xr, c, h * w), (dy, dyr, k, pixels))):
        call(lib.sd_conv2d_taps_prepare, 1, array(C.c_void_p, src.data_ptr()), array(C.c_int64, src.stride(0)), array(C.c_int64, src.stride(1)),
             array(C.c_void_p, dst.data_ptr()), array(C.c_int64, n), array(C.c_int64, ch), array(C.c_int64, px), wt.data_ptr(), c * r * s,
             c, k, r, s, b, packed[b].data_ptr(), None, 0, 0, None, 0, 0, 0.0, dt, st)
    m = mask.cuda() if mask is not None else None
    ms = (m.data_ptr(), m.stride(0), m.stride(1), bs) if mask is not None else (None, 0, 0, 0)
    call(lib.sd_conv2d_taps_forward, xr.data_ptr(), c, packed[0].data_ptr(), y.data_ptr(), k, *ms, *geo, scale, dt, st)
    dx = torch.full((n, c, h, w), 77.0, dtype=x.dtype, device="cuda")
    if channels_last:
        dx = dx.contiguous(memory_format=torch.channels_last)
    call(lib.sd_conv2d_taps_dx, dyr.data_ptr(), k, packed[1].data_ptr(), dx.data_ptr(), *dx.stride(), *ms, *geo, scale, dt, st)
    ws = torch.empty(lib.sd_conv2d_taps_dw_workspace_bytes(c, k, r, s, rows), dtype=torch.uint8, device="cuda")
    call(lib.sd_conv2d_taps_dw, xr.data_ptr(), c, dyr.data_ptr(), k, dw.data_ptr(), c * r * s, *ms, *geo, scale, dt, ws.data_ptr(),
         ws.numel(), st)
    return y.view(n, dy.shape[2], dy.shape[3], k).permute(0, 3, 1, 2), dx, dw.view(k, c, r, s)


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("bs,p", [(64, 0.5), (128, 0.3), (0, 0.0)])
@pytest.mark.parametrize("channels_last", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_products_tap_by_tap(geom, bs, p, channels_last, dtype):
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, dtype)
    mask = cpu_mask(O.mask_shape(rows, c * r * s, bs or 64), p, gen)
    args = (geom, x, wt, dy, mask if bs else None, bs, 1 / (1 - p), channels_last)
    got = _products(*args)
    geo = dict(padding=pad, stride=(1, 1), dilation=dil)
    want = O.conv2d_blockdrop(to_np(x), to_np(wt), mask.numpy(), bs or 64, p, dy=to_np(dy), dtype=np.float64, **geo)
    for g, ref in zip(got, want):
        assert max_tile_rel_fro(g, ref) <= REL_FRO_TOL
    # the same bits once more: every sum has one owner and one order
    assert all(torch.equal(a, b) for a, b in zip(got, _products(*args)))


# channels, outputs: last groups of 8 to 128 outputs (of 64 channels in the input gradient) and last chunks of one slab and of two,
# first groups and chunks in front of them and not
@pytest.mark.parametrize("c,k", [(72, 72), (96, 88), (104, 96), (40, 104), (64, 136), (160, 160), (168, 184), (224, 232), (128, 256),
                                 (88, 32), (24, 80), (136, 24)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs,p,channels_last", [(64, 0.4, False), (0, 0.0, True)])
def test_channels_that_end_inside_a_tile_group(c, k, dtype, bs, p, channels_last):
    geom = (3, c, 10, 13, k, 3, 3, (1, 1), (1, 1))
    x, wt, dy, rows, gen = _tensors(geom, dtype, seed=c + k)
    mask = cpu_mask(O.mask_shape(rows, c * 9, bs or 64), p, gen)
    got = _products(geom, x, wt, dy, mask if bs else None, bs, 1 / (1 - p), channels_last)
    want = O.conv2d_blockdrop(to_np(x), to_np(wt), mask.numpy(), bs or 64, p, dy=to_np(dy), dtype=np.float64, padding=(1, 1),
                              stride=(1, 1), dilation=(1, 1))
    for g, ref in zip(got, want):
        assert max_tile_rel_fro(g, ref) <= REL_FRO_TOL


# (geometry, channels-last image, whether the image is what is kept): rows that fill blocks of 64 and rows that do not
LAYERS = [((20, 24, 16, 16, 40, 3, 3, (1, 1), (1, 1)), False, True), ((20, 32, 16, 16, 40, 3, 3, (1, 1), (1, 1)), True, False),
          ((7, 16, 28, 28, 40, 3, 3, (1, 1), (1, 1)), False, False), ((7, 16, 28, 28, 40, 5, 5, (2, 2), (1, 1)), True, False)]


@pytest.mark.parametrize("geom,channels_last,keeps_image", LAYERS)
@pytest.mark.parametrize("drawn", [False, True])
def test_layers_tap_by_tap(geom, channels_last, keeps_image, drawn):
    """The autograd function on this route: results, what is kept, and which changes before the backward are refused."""
    import flash_dropout.functional as F
    from flash_dropout.hip import GEMM

    n, c, h, w, k, r, s, pad, dil = geom
    assert GEMM().lib.sd_conv2d_taps_taken(n, c, h, w, k, r, s, *pad, 1, 1, *dil, 0.4) == 1
    x, wt, dy, rows, gen = _tensors(geom, torch.float16)
    shape = O.mask_shape(rows, c * r * s, 64)
    mask = torch.from_numpy(O.random_mask(shape, 0.4, 5)) if drawn else cpu_mask(shape, 0.4, gen)
    xg = x.cuda()
    if channels_last:
        xg = xg.contiguous(memory_format=torch.channels_last)
    xg.requires_grad_()
    wg = wt.cuda().requires_grad_()
    call = lambda: (F.blockwise_dropout_conv2d(xg, wg, 64, 0.4, pad, seed=5) if drawn else
                    F.blockwise_dropout_conv2d_mask(xg, mask.cuda(), 64, 0.4, wg, pad))
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
        call()
    big = [q for q in kept if len(q) == 4 or q[0] >= 4096]
    assert big == [tuple(x.shape) if keeps_image else (n * h * w, c)]
    y = call()
    grads = torch.autograd.grad(y, (xg, wg), dy.cuda(), retain_graph=True)
    assert F.conv_last_routes() == {"forward": "implicit", "dx": "fused", "dw": "implicit"}
    assert grads[0].stride() == xg.stride()
    want = O.conv2d_blockdrop(to_np(x), to_np(wt), mask.numpy(), 64, 0.4, dy=to_np(dy), dtype=np.float64, padding=pad, stride=(1, 1),
                              dilation=dil)
    for g, ref in zip((y.detach(), *grads), want):
        assert max_tile_rel_fro(g, ref) <= REL_FRO_TOL
    with torch.no_grad():
        xg.mul_(2)
    if keeps_image:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(y, (xg, wg), dy.cuda())
    else:
        again = torch.autograd.grad(y, (xg, wg), dy.cuda())
        assert all(torch.equal(a, b) for a, b in zip(again, grads))


def test_rows_are_kept_for_the_kernel_gradient_only():
    """Where the rows and not the image are what the kernel's gradient reads: a frozen kernel keeps neither, the image may change
    before the backward as it may otherwise, and dX is the same."""
    import flash_dropout.functional as F

    geom = LAYERS[1][0]
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, torch.float16)
    xg = x.cuda().contiguous(memory_format=torch.channels_last).requires_grad_()
    wg = wt.cuda().requires_grad_()
    both = torch.autograd.grad(F.blockwise_dropout_conv2d(xg, wg, 64, 0.4, pad, seed=5), (xg, wg), dy.cuda())
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
        y = F.blockwise_dropout_conv2d(xg, wg.detach(), 64, 0.4, pad, seed=5)
    assert [q for q in kept if len(q) == 4 or q[0] >= 4096] == []
    with torch.no_grad():
        xg.mul_(2)
    assert torch.equal(torch.autograd.grad(y, xg, dy.cuda())[0], both[0])


@pytest.mark.parametrize("sliced", ["channels", "channels off 16 bytes", "channels at an odd distance", "pixels", "planes"])
def test_slices_tap_by_tap(sliced):
    """Images and gradients that are slices: their own rows, copied once, or turned, they give the same bits as whole ones."""
    import flash_dropout.functional as F

    geom = (20, 32, 16, 16, 40, 3, 3, (1, 1), (1, 1))
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, torch.float16)

    def slice_of(t):
        b, ch, p, q = t.shape
        cl = dict(memory_format=torch.channels_last)
        wide, at = {"channels": ((b, 2 * ch, p, q), (0, ch, 0, 0)), "channels off 16 bytes": ((b, 2 * ch, p, q), (0, 4, 0, 0)),
                    "channels at an odd distance": ((b, ch + 4, p, q), (0, 0, 0, 0)), "pixels": ((b, ch, p + 2, q + 3), (0, 0, 1, 2)),
                    "planes": ((b, ch, p + 2, q + 3), (0, 0, 1, 2))}[sliced]
        big = torch.randn(wide, dtype=t.dtype, device="cuda")
        big = big.contiguous(**({} if sliced == "planes" else cl))
        view = big[tuple(slice(o, o + e) for o, e in zip(at, t.shape))]
        return view.copy_(t)

    def products(xg, dyg):
        xg, wg = xg.detach().requires_grad_(), wt.cuda().requires_grad_()
        y = F.blockwise_dropout_conv2d(xg, wg, 64, 0.4, pad, seed=5)
        return (y, *torch.autograd.grad(y, (xg, wg), dyg))

    whole = products(x.cuda(), dy.cuda())
    for xg, dyg in ((slice_of(x), dy.cuda()), (x.cuda(), slice_of(dy)), (slice_of(x), slice_of(dy))):
        assert all(torch.equal(a, b) for a, b in zip(products(xg, dyg), whole))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_what_a_mask_drops_reaches_nothing_tap_by_tap(bad):
    """An Inf or NaN in an operand reaches the results whose kept blocks read it, and no other."""
    geom = (3, 32, 14, 14, 64, 3, 3, (1, 1), (1, 1))
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, torch.float16)
    mask = cpu_mask(O.mask_shape(rows, c * r * s, 64), 0.5, gen)
    keep = ~mask.repeat_interleave(64, 0).repeat_interleave(64, 1)[:rows, : c * r * s]
    for which in range(3):
        ops = [t.clone() for t in (x, wt, dy)]
        ops[which].view(-1)[ops[which].numel() // 3] = bad
        y, dx, dw = _products(geom, *ops, mask, 64, 2.0)
        # counted over kept elements only: where a bad value is not among a sum's terms, the sum is finite
        cols = torch.nn.functional.unfold(ops[0].double(), (r, s), padding=pad).permute(0, 2, 1).reshape(rows, -1)
        wm, dm = ops[1].double().reshape(k, -1), ops[2].double().permute(0, 2, 3, 1).reshape(rows, k)
        b_cols, b_w, b_dy = (~torch.isfinite(t) for t in (cols, wm, dm))
        kf = keep.double()
        bad_y = ((b_cols & keep).double() @ torch.ones(c * r * s, k, dtype=torch.double) + kf @ b_w.double().T) > 0
        bad_cols = keep & ((b_dy.double() @ torch.ones(k, c * r * s, dtype=torch.double) +
                            torch.ones(rows, k, dtype=torch.double) @ b_w.double()) > 0)
        bad_dx = torch.nn.functional.fold(bad_cols.double().reshape(n, h * w, -1).permute(0, 2, 1), (h, w), (r, s), padding=pad) > 0
        bad_dw = (b_dy.double().T @ kf + torch.ones(k, rows, dtype=torch.double) @ (b_cols & keep).double()) > 0
        assert torch.equal(~torch.isfinite(y.permute(0, 2, 3, 1).reshape(rows, k).cpu()), bad_y), which
        assert torch.equal(~torch.isfinite(dx.cpu()), bad_dx), which
        assert torch.equal(~torch.isfinite(dw.cpu().reshape(k, -1)), bad_dw), which


def _dw_turns(geom):
    """Least and most turns of 256 positions that a workgroup of the weight gradient has."""
    from flash_dropout.hip import GEMM

    n, c, h, w, k, r, s, pad, dil = geom
    rows = n * h * w  # (as many positions as pixels)
    turns, parts = -(-rows // 256), GEMM().lib.sd_conv2d_taps_dw_workspace_bytes(c, k, r, s, rows) // (4 * c * k * r * s)
    return turns // parts, -(-turns // parts)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("geom,turns", [
    ((1, 512, 12, 256, 256, 3, 3, (1, 1), (1, 1)), (3, 3)),  # a window of 784 rows: the only buffer is filled again
    ((2, 264, 11, 256, 232, 3, 3, (1, 1), (1, 1)), (3, 4)),  # parts of uneven length, channels and outputs that end inside a tile
    ((3, 512, 24, 40, 200, 3, 3, (1, 1), (1, 1)), (3, 3)),    # two, the first of them used twice, the last turn not whole
])
def test_weight_gradient_over_several_turns(geom, turns, dtype):
    assert _dw_turns(geom) == turns
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, dtype)
    mask = cpu_mask(O.mask_shape(rows, c * r * s, 64), 0.5, gen)
    dw = _products(geom, x, wt, dy, mask, 64, 2.0)[2]
    want = O.conv2d_blockdrop(to_np(x), to_np(wt), mask.numpy(), 64, 0.5, dy=to_np(dy), dtype=np.float32, padding=pad, stride=(1, 1),
                              dilation=dil)[2]
    assert max_tile_rel_fro(dw, want) <= REL_FRO_TOL


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("geom,turns", [
    ((16, 128, 32, 32, 128, 3, 3, (1, 1), (1, 1)), (2, 2)),
    ((2, 512, 24, 40, 200, 3, 3, (1, 1), (1, 1)), (2, 2)),    # the last turn not whole
    ((3, 512, 24, 40, 200, 3, 3, (1, 1), (1, 1)), (3, 3)),
    ((1, 32, 9, 256, 40, 3, 3, (1, 1), (1, 1)), (1, 1)),    # one buffer
    ((1, 512, 12, 256, 256, 3, 3, (1, 1), (1, 1)), (3, 3)),
])
def test_gradients_that_are_not_finite_reach_kept_blocks_only(geom, turns, bad):
    """A weight gradient clears what a block drops in the image, and does without where a sum is not finite: one bad element of dY
    reaches its output's kept blocks, and everything else is bit for bit what it is with a zero there.  The turns are gone through
    a second time for that, with one and with two buffers for their rows."""
    assert _dw_turns(geom) == turns
    n, c, h, w, k, r, s, pad, dil = geom
    x, wt, dy, rows, gen = _tensors(geom, torch.float16)
    mask = cpu_mask(O.mask_shape(rows, c * r * s, 64), 0.5, gen)
    at = rows // 2 + 7, k // 3
    img, pos = divmod(at[0], rows // n)
    got = []
    for v in (0.0, bad):
        dy.view(n, k, -1)[img, at[1], pos] = v
        got.append(_products(geom, x, wt, dy, mask, 64, 2.0)[2].cpu().reshape(k, -1))
    reached = torch.zeros(k, c * r * s, dtype=torch.bool)
    reached[at[1]] = ~mask[at[0] // 64].repeat_interleave(64)[: c * r * s]
    assert torch.equal(~torch.isfinite(got[1]), reached)
    assert torch.equal(got[1][~reached], got[0][~reached])


@pytest.mark.parametrize("geom", [
    (256, 32, 28, 28, 64, 3, 3, (1, 1), (1, 1)),  # 784 turns in 256 parts, three or four each
    (24, 64, 32, 32, 64, 3, 3, (1, 1), (1, 1)),   # 96 in 96 of at most 128
    (35, 72, 16, 20, 200, 3, 3, (1, 1), (1, 1)),  # 44 in 21
])
def test_order_in_which_a_weight_gradients_parts_are_added_up(geom):
    """Bit for bit: as many parts as fill the chip once, sixteen chains, chain j the parts j, j + 16, ... in order, then the chains in
    order.  Every part holds one exact product at the middle tap, 2^25, its negative or a small integer, whose fp32 sums
    depend on the order."""
    n, c, h, w, k, r, s, pad, dil = geom
    rows, gen = n * h * w, torch.Generator().manual_seed(k)
    turns, tiles = -(-rows // 256), -(-c // 32) * -(-k // 64)
    parts = min(256 // tiles, turns)
    first = [i * (turns // parts) + min(i, turns % parts) for i in range(parts)]
    values = torch.randint(-15, 16, (parts, k), generator=gen).float()
    for j in range(k):
        at = torch.randperm(parts, generator=gen)[: parts // 4 * 2]
        values[at, j] = 2.0 ** 25 * (1.0 - 2.0 * (torch.arange(len(at)) % 2))
    x, dy = torch.zeros(n, c, h * w).half(), torch.zeros(n, k, h * w).half()
    for i, turn in enumerate(first):
        img, at = divmod(turn * 256 + 100, h * w)
        x[img, :, at] = 1024.0
        dy[img, :, at] = (values[i] / 1024.0).half()
    wt = torch.zeros(k, c, r, s).half()
    mask = torch.zeros(O.mask_shape(rows, c * r * s, 64), dtype=torch.bool)
    dw = _products(geom, x.view(n, c, h, w), wt, dy.view(n, k, h, w), mask, 64, 1.0)[2].cpu().reshape(k, c, r * s)
    def in_order(terms):
        total = torch.zeros(k)
        for t in terms:
            total = total + t
        return total
    want = in_order([in_order(values[j::16]) for j in range(16)])
    for other in (in_order(values), in_order([in_order(values[j::64]) for j in range(64)])):
        assert not torch.equal(want, other)
    assert torch.equal(dw[:, :, 4].float(), want[:, None].expand(k, c))
