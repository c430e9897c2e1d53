"""Which workgroup has which column blocks in the input gradient: row quads dealt out to groups at the edges of the rule, groups
and strips by a hint that is right or far off, and positions counted over all row quads."""
import pytest
import torch

from _util import max_tile_rel_fro

pytestmark = pytest.mark.gpu

# column blocks of a row quad with one or two kept tiles, and with three or four
DEALS = [(0, 0), (1, 0), (0, 1), (6, 0), (7, 0), (0, 4), (0, 5), (4, 2), (5, 2), (3, 9), (13, 3), (12, 4), (66, 1), (1, 66), (24, 40),
         (0, 96), (96, 0), (47, 49), (2, 8), (11, 7)]


def quad_rows(n1, n2, Cb, gen):
    """Keep bits of four row blocks with n1 and n2 such columns at random places."""
    keep = torch.zeros(4, Cb, dtype=torch.bool)
    for i, c in enumerate(torch.randperm(Cb, generator=gen)[: n1 + n2].tolist()):
        k = (1 + i % 2) if i < n1 else (3 + i % 2)
        keep[torch.randperm(4, generator=gen)[:k], c] = True
    return keep


def check(ext, dy, w, mask, p, hint, policy, bs=64):
    """dX against fp32 on the same rounded operands: one rounding to fp16 is 2^-11 of an element at most, and a sum of K products
    in fp32 adds K * 2^-24 of the terms' size, so 2^-10 of a tile's norm holds both."""
    lists = ext.build_lists(mask, 0 if bs == 32 else 1)
    M, N = dy.shape[0], w.shape[1]
    out = torch.full((M, N), 7.0, dtype=dy.dtype, device="cuda")
    before = ext.set_tile_policy(policy)
    try:
        ext.gemm_sdd_lists(dy, w.t(), lists, bs, 1.0 / (1.0 - p), out=out, keep_hint=hint)
        detail = ext.last_kernel_detail()
    finally:
        ext.set_tile_policy(before)
    keep = (~mask).repeat_interleave(bs, 0)[:M].repeat_interleave(bs, 1)[:, :N]
    ref = (dy.float() @ w.float()) / (1.0 - p) * keep
    assert max_tile_rel_fro(out, ref) <= 2.0 ** -10
    return detail


@pytest.mark.parametrize("hint", [None, 0.9, 0.5, 0.02])
@pytest.mark.parametrize("N", [96 * 64, 96 * 64 - 24])
@pytest.mark.parametrize("policy", ["big", "mid"])
def test_rows_dealt_out_to_groups(N, hint, policy):
    from flash_dropout.hip import GEMM

    gen = torch.Generator().manual_seed(N)
    mask = ~torch.cat([quad_rows(*d, 96, gen) for d in DEALS])[: 4 * len(DEALS) - 1]  # the last quad has three row blocks
    M, K = 64 * mask.shape[0] - 3, 256
    dy, w = torch.randn(M, K, generator=gen).half().cuda(), torch.randn(K, N, generator=gen).half().cuda()
    detail = check(GEMM(), dy, w, mask.cuda(), 0.5, hint, policy)
    assert detail.startswith("sdd:" + policy)


@pytest.mark.parametrize("M,N,K,p,bs,counted", [
    (2048, 24320, 3072, 0.5, 64, True),    # 8 row quads
    (2304, 22056, 3080, 0.5, 64, True),    # 9, ragged column blocks and steps
    (12288, 3584, 3072, 0.8, 32, True),    # 48, masks of 32-blocks
    (33280, 1344, 3072, 0.5, 64, True),    # 130: a thread to a row of blocks, two turns of them
    (65530, 576, 3072, 0.5, 64, True),     # 256, the most that are counted, the last row block not whole
    (65600, 576, 3072, 0.5, 64, False),    # 257
    (2048, 24320, 3008, 0.5, 64, False),   # 47 steps
    (12288, 1088, 512, 0.3, 64, False),    # three quarters of a round
    (4096, 4096, 256, 0.5, 64, False),
])
def test_positions_counted_over_all_row_quads(M, N, K, p, bs, counted):
    from flash_dropout.hip import GEMM

    gen = torch.Generator(device="cuda").manual_seed(M + N)
    dy = torch.randn(M, K, generator=gen, device="cuda").half()
    w = torch.randn(K, N, generator=gen, device="cuda").half()
    mask = torch.rand(-(-M // bs), -(-N // bs), generator=gen, device="cuda") < p
    mask[: 512 // bs, ::2] = True  # quads with fewer groups than the others
    detail = check(GEMM(), dy, w, mask, p, 1.0 - p, "big", bs)
    assert detail.startswith("sdd:big") and detail.endswith(":counted") == counted, detail


def test_positions_are_not_counted_beside_the_weight_gradient():
    """The weight gradient's workgroups fill the last round there: the pair's dX has the bits of the launch alone, whichever way
    its positions are found."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    M, N, K, p, bs = 65280, 768, 3072, 0.75, 64  # 255 row quads
    gen = torch.Generator(device="cuda").manual_seed(M)
    x, w, dy = (torch.randn(*s, generator=gen, device="cuda").half() for s in ((M, N), (K, N), (M, K)))
    mask = torch.rand(M // bs, N // bs, generator=gen, device="cuda") < p
    before = ext.set_tile_policy("big")
    try:
        _, _, lists, kbs = ext.dropout_matmul_forward(x, w, bs, p, mask=mask)
        dx, _ = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p)
        pair = ext.last_kernel_detail()
        alone, _ = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p, need_dw=False)
        assert ext.last_kernel_detail() == "sdd:big:counted"
    finally:
        ext.set_tile_policy(before)
    assert pair.startswith("pair:sdd+dsd:big") and "counted" not in pair, pair
    assert torch.equal(dx, alone)


@pytest.mark.parametrize("bs", [32, 64])
def test_groups_beside_the_weight_gradient(bs):
    """Both gradients in one launch on the big shape, masks of 32-blocks included, against the two launches."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    M, N, K, p = 1536, 512, 2048, 0.6
    gen = torch.Generator(device="cuda").manual_seed(bs)
    x, w, dy = (torch.randn(*s, generator=gen, device="cuda").half() for s in ((M, K), (N, K), (M, N)))
    mask = torch.rand(M // bs, K // bs, generator=gen, device="cuda") < p
    before = ext.set_tile_policy("big")
    try:
        _, _, lists, kbs = ext.dropout_matmul_forward(x, w, bs, p, mask=mask)
        dx, _ = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p)
        assert ext.last_kernel_detail().startswith("pair:sdd+dsd:big")
        alone, _ = ext.dropout_matmul_backward(dy, w, x, lists, kbs, p, need_dw=False)
    finally:
        ext.set_tile_policy(before)
    keep = (~mask).repeat_interleave(bs, 0).repeat_interleave(bs, 1)
    assert torch.equal(dx, alone) and max_tile_rel_fro(dx, (dy.float() @ w.float()) / (1 - p) * keep) <= 2.0 ** -10
