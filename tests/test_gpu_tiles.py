"""The 64 x 64 and 128 x 128 tile kernels at the sizes where they can go wrong: one step, fewer steps than stages, one more
than a full round of stages, ragged last blocks in every extent, widths that are not multiples of 8, row blocks and
tiles without a kept block, quadrant masks, split reductions."""
import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, cpu_mask, make_operand, max_tile_rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,bs,p", [
    (64, 64, 64, 64, 0.0),         # one workgroup, one step
    (65, 72, 72, 64, 0.4),         # one past a tile everywhere
    (127, 136, 200, 64, 0.5),      # fewer steps than stages, ragged last step
    (190, 200, 328, 32, 0.6),      # quadrant keep bits, ragged everywhere
    (1, 8, 264, 64, 0.3),          # a single row
    (300, 1096, 1032, 64, 0.95),   # row blocks with nothing kept; the first extent past the 64 x 64 shape's round
    (1100, 1288, 520, 96, 0.3),    # 128 x 128 tiles, an odd multiple of 32
    (2200, 2056, 136, 64, 0.2),    # more than a round of 128 x 128 tiles
    (72, 200, 16456, 64, 0.5),     # long reduction, few tiles: split in the forward and in the weight gradient
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_products_on_the_tile_shapes(M, N, K, bs, p, dtype):
    """Forward, dX and dW of a layer X[M, K] -> N against the fp32 oracle on the same rounded operands, per 64-tile.
    The bar is the suite's relative Frobenius one; sums are fp32 and rounded once, so it has orders of magnitude of room."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K + bs)
    x = make_operand(M, K, dtype, "cuda", gen=gen)
    w = make_operand(N, K, dtype, "cuda", scale=K ** -0.5, gen=gen)
    dy = make_operand(M, N, dtype, "cuda", gen=gen)
    mask = cpu_mask(O.mask_shape(M, K, bs), p, gen)
    mk = mask.numpy()
    y, _, lists, kbs = ext.dropout_matmul_forward(x, w, bs, p, mask=mask.cuda())
    assert ext.last_kernel() == "specialised"
    dx, dw = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p)
    assert ext.last_kernel() == "specialised"
    xn, wn, dyn = to_np(x), to_np(w), to_np(dy)
    for got, ref, what in ((y, O.dsd_forward(xn, wn, mk, bs, p, np.float32), "y"),
                           (dx, O.sdd_dx(dyn, wn, mk, bs, p, np.float32), "dx"),
                           (dw, O.dsd_dw(dyn, xn, mk, bs, p, np.float32), "dw")):
        assert max_tile_rel_fro(got, ref) <= REL_FRO_TOL, what
    keep = O.expand_keep(mk, bs, M, K)
    assert (dx.float().cpu().numpy()[~keep] == 0).all()


@pytest.mark.parametrize("M,N,K", [(64, 13, 64), (200, 77, 136), (515, 301, 264)])
@pytest.mark.parametrize("act", ["relu", "gelu"])
def test_unaligned_output_rows(M, N, K, act):
    """Output rows that start at any 2-byte boundary (N odd), with the activation and its pre-activation in the store;
    kept-only and zeroed SDD tiles into such rows."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(M + N)
    x = make_operand(M, K, torch.float16, "cuda", gen=gen)
    w = make_operand(N, K, torch.float16, "cuda", scale=K ** -0.5, gen=gen)
    mask = cpu_mask(O.mask_shape(M, K, 64), 0.4, gen)
    lists = ext.build_lists(mask.cuda())
    got, pre = ext.gemm_dsd_lists_act(x, w, lists, 64, 2.0, act, want_pre=True)
    assert ext.last_kernel() == "specialised"
    ref = O.gemm_dsd(to_np(x), to_np(w), mask.numpy(), 64, 2.0, np.float32)
    assert max_tile_rel_fro(pre, ref) <= REL_FRO_TOL
    t = torch.from_numpy(np.asarray(ref))
    assert max_tile_rel_fro(got, (torch.relu(t) if act == "relu" else torch.nn.functional.gelu(t)).numpy()) <= REL_FRO_TOL
    # SDD into odd rows: B is [N, K] with its reduction index strided, in rows wide enough for 16-byte loads
    wide = torch.randn(K, -(-N // 8) * 8, generator=gen).half().cuda()
    b = wide[:, :N].t()
    mask = cpu_mask(O.mask_shape(M, N, 64), 0.5, gen)
    lists = ext.build_lists(mask.cuda())
    out = torch.full((M, N), 7.0, dtype=torch.float16, device="cuda")
    ext.gemm_sdd_lists(x, b, lists, 64, 0.5, out=out)
    assert ext.last_kernel() == "specialised"
    assert max_tile_rel_fro(out, O.gemm_sdd(to_np(x), to_np(b), mask.numpy(), 64, 0.5, np.float32)) <= REL_FRO_TOL
    assert (out.cpu().numpy()[~O.expand_keep(mask.numpy(), 64, M, N)] == 0).all()


@pytest.mark.parametrize("act", [None, "gelu"])
def test_input_gradient_of_a_short_reduction(act):
    """A grid of one and a half rounds of the big shape, which strips of two take over.  Reference in fp32 on the same
    rounded operands; one rounding to bf16 (2^-9 relative on average of at most 2^-8)."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    M, C, K = 4096, 6144, 264
    gen = torch.Generator(device="cuda").manual_seed(1)
    dy, w, at = (torch.randn(*s, generator=gen, device="cuda").bfloat16() for s in ((M, K), (K, C), (M, C)))
    mask = torch.rand(M // 64, C // 64, generator=gen, device="cuda") < 0.5
    lists = ext.build_lists(mask)
    for k in (256, K):  # aligned reduction; a ragged one, which stays where it was
        a, b = dy[:, :k].contiguous(), w[:k].contiguous()
        if act:
            got = ext.gemm_sdd_lists_actgrad(a, b.t(), lists, 64, 2.0, act, at, keep_hint=0.5)
        else:
            got = ext.gemm_sdd_lists(a, b.t(), lists, 64, 2.0, keep_hint=0.5)
        assert k != 256 or ext.last_kernel_detail() == "sdd:mid"
        ref = 2.0 * (a.float() @ b.float())
        if act:
            t = at.float()
            ref *= 0.5 * (1 + torch.erf(t * 0.5 ** 0.5)) + t * torch.exp(-0.5 * t * t) * 0.3989422804014327
        ref *= (~mask).repeat_interleave(64, 0).repeat_interleave(64, 1)
        assert (got[ref == 0] == 0).all() and (got.float() - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("M,N,K,bs", [
    (32832, 50, 200, 64),   # one tile past the 512 that are resident, a ragged last step
    (33001, 64, 64, 32),    # fewer steps than stages, quadrant keep bits
    (34000, 61, 520, 64),   # more steps than stages, an odd width
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_more_small_tiles_than_are_resident(M, N, K, bs, dtype):
    """The forward on the three-stage 64 x 64 shape, with the lists in the same launch and from lists, and dense."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(K)
    x = make_operand(M, K, dtype, "cuda", gen=gen)
    w = make_operand(N, K, dtype, "cuda", scale=K ** -0.5, gen=gen)
    mask = cpu_mask(O.mask_shape(M, K, bs), 0.4, gen)
    y, _, lists, kbs = ext.dropout_matmul_forward(x, w, bs, 0.4, mask=mask.cuda())
    again = ext.gemm_dsd_lists(x, w, lists, kbs, 1 / 0.6)
    assert ext.last_kernel_detail().startswith("dsd:one")
    ref = O.dsd_forward(to_np(x), to_np(w), mask.numpy(), bs, 0.4, np.float32)
    assert max_tile_rel_fro(y, ref) <= REL_FRO_TOL and torch.equal(y, again)
    assert max_tile_rel_fro(ext.gemm(x, w), to_np(x) @ to_np(w).T) <= REL_FRO_TOL


@pytest.mark.parametrize("M,C,N,bs,shape", [
    (65, 72, 64, 64, "auto"),       # strips of one: one past a tile, one step
    (200, 61, 264, 32, "auto"),     # an odd width, whose last eight are stored one by one; quadrant bits
    (4096, 6144, 256, 64, "auto"),  # strips of two
    (530, 1029, 136, 64, "big"),    # groups of the large shape, ragged everywhere
])
@pytest.mark.parametrize("act", ["relu", "gelu"])
def test_pre_activations_of_any_rows(M, C, N, bs, shape, act):
    """The derivative at pre-activations that lie in rows of their own pitch and start, off every boundary: the bits of the
    same ones in aligned rows, which are held to fp32 (one rounding to bf16, at most 2^-8 relative)."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator(device="cuda").manual_seed(M + C)
    pad = -C % 8
    dy = torch.randn(M, N, generator=gen, device="cuda").bfloat16()
    w = torch.randn(N, C + pad, generator=gen, device="cuda").bfloat16()[:, :C]
    at = torch.randn(M, C, generator=gen, device="cuda").bfloat16()
    apart = torch.full((M, C + 3), float("nan"), dtype=torch.bfloat16, device="cuda")
    apart[:, 1:1 + C] = at
    mask = torch.rand(-(-M // bs), -(-C // bs), generator=gen, device="cuda") < 0.4
    lists, kbs = (ext.build_lists(mask, 0 if bs == 32 else 1), bs)
    before = ext.set_tile_policy(shape)
    try:
        got, other = (ext.gemm_sdd_lists_actgrad(dy, w.t(), lists, kbs, 1.5, act, a, keep_hint=0.6)
                      for a in (at, apart[:, 1:1 + C]))
    finally:
        ext.set_tile_policy(before)
    assert torch.equal(got, other)
    t = at.float()
    d = (t > 0).float() if act == "relu" else 0.5 * (1 + torch.erf(t * 0.5 ** 0.5)) + t * torch.exp(-0.5 * t * t) * 0.3989422804014327
    keep = (~mask).repeat_interleave(bs, 0)[:M].repeat_interleave(bs, 1)[:, :C]
    ref = 1.5 * (dy.float() @ w.float()) * d * keep
    assert (got[~keep] == 0).all() and (got.float() - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("M,K,N,bs,p,shape", [
    (2048, 200, 136, 64, 0.5, "one"),    # the weight gradient's chains are longer, its 12 workgroups no multiple of 8
    (136, 200, 2056, 64, 0.5, "one"),    # the input gradient's
    (1032, 1024, 784, 32, 0.6, "one"),   # about as long
    (4040, 2048, 1000, 64, 0.1, "mid"),
    (2048, 1096, 3064, 64, 0.25, "mid"),
])
def test_both_gradients_in_one_launch_in_either_order(M, K, N, bs, p, shape):
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(M + N + K)
    x = make_operand(M, K, torch.float16, "cuda", gen=gen)
    w = make_operand(N, K, torch.float16, "cuda", scale=K ** -0.5, gen=gen)
    dy = make_operand(M, N, torch.float16, "cuda", gen=gen)
    mask = cpu_mask(O.mask_shape(M, K, bs), p, gen)
    _, _, lists, kbs = ext.dropout_matmul_forward(x, w, bs, p, mask=mask.cuda())
    dx, dw = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p)
    assert ext.last_kernel_detail().startswith("pair:sdd+dsd:" + shape), ext.last_kernel_detail()
    mk = mask.numpy()
    assert max_tile_rel_fro(dx, O.sdd_dx(to_np(dy), to_np(w), mk, bs, p, np.float32)) <= REL_FRO_TOL
    assert max_tile_rel_fro(dw, O.dsd_dw(to_np(dy), to_np(x), mk, bs, p, np.float32)) <= REL_FRO_TOL
