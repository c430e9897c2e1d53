"""Which workgroup shape large and ragged products run on, and the cuts of the reduction that go with it."""
import numpy as np
import pytest
import torch

from _util import REL_FRO_TOL, cpu_mask, make_operand, max_tile_rel_fro, to_np
from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu


def _layer(M, K, N, bs, p, dtype):
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(M + K + N)
    x, dy = make_operand(M, K, dtype, "cuda", gen=gen), make_operand(M, N, dtype, "cuda", gen=gen)
    w = make_operand(N, K, dtype, "cuda", scale=K ** -0.5, gen=gen)
    mask = cpu_mask(O.mask_shape(M, K, bs), p, gen)
    _, lists, kbs = ext.kept_lists(M, K, bs, mask=mask.cuda())
    return ext, x, w, dy, mask.numpy(), lists, kbs


@pytest.mark.parametrize("M,K,N,bs,p", [
    (4224, 4800, 2048, 128, 0.05),  # 160 us forward on the 64 x 64 shape, 99 on the big one
    (3520, 6912, 1728, 128, 0.3),   # 131 and 87
    (9664, 7808, 512, 32, 0.4),     # 181 and 92 on 128 x 128 tiles
])
def test_large_forward_products_leave_the_smallest_shape(M, K, N, bs, p):
    ext, x, w, _, mk, lists, kbs = _layer(M, K, N, bs, p, torch.float16)
    y = ext.gemm_dsd_lists(x, w, lists, kbs, 1 / (1 - p))
    assert ext.last_kernel() == "specialised" and not ext.last_kernel_detail().startswith("dsd:one"), ext.last_kernel_detail()
    assert max_tile_rel_fro(y, O.dsd_forward(to_np(x), to_np(w), mk, bs, p, np.float32)) <= REL_FRO_TOL


@pytest.mark.parametrize("M,K,N,bs,p,dtype,cut", [
    (13888, 2840, 3472, 32, 0.1, torch.float16, False),   # 1124 us on the 64 x 64 shape
    (13568, 1536, 3264, 64, 0.25, torch.bfloat16, True),  # whole blocks, the big shape in several parts
    (10368, 200, 6352, 64, 0.5, torch.float16, True),     # 128 x 128 tiles without loading waves, several parts
    (9024, 864, 5549, 64, 0.25, torch.bfloat16, False),   # the same with an output width that is no multiple of 8
])
def test_large_weight_gradients_leave_the_smallest_shape(M, K, N, bs, p, dtype, cut):
    ext, x, _, dy, mk, lists, kbs = _layer(M, K, N, bs, p, dtype)
    if N % 8:  # as the autograd functions do: zero columns up to the next multiple
        dy = torch.nn.functional.pad(dy, (0, -N % 8))
    dw = ext.gemm_dsd_lists(x.t(), dy.t(), lists.transposed(), kbs, 1 / (1 - p), transposed_out=True).t()[:N]
    detail = ext.last_kernel_detail()
    assert ext.last_kernel() == "specialised" and not detail.startswith("dsd:one"), detail
    assert detail.endswith("splits=1") != cut, detail
    assert max_tile_rel_fro(dw, O.dsd_dw(to_np(dy)[:, :N], to_np(x), mk, bs, p, np.float32)) <= REL_FRO_TOL


@pytest.mark.parametrize("M,K,N,p,act", [
    (6574, 4808, 5704, 0.5, None),    # 592 us on strips of two, 338 on the big shape's edge instance
    (6656, 6736, 7008, 0.1, "gelu"),  # 1474 and 635
])
def test_large_ragged_input_gradients_stay_on_the_big_shape(M, K, N, p, act):
    ext, x, w, dy, mk, lists, kbs = _layer(M, K, N, 64, p, torch.float16)
    s = 1 / (1 - p)
    if act:
        dx = ext.gemm_sdd_lists_actgrad(dy, w.t(), lists, kbs, s, act, x, keep_hint=1 - p)
    else:
        dx = ext.gemm_sdd_lists(dy, w.t(), lists, kbs, s, keep_hint=1 - p)
    assert ext.last_kernel_detail() == "sdd:big:ragged", ext.last_kernel_detail()
    ref = O.sdd_dx(to_np(dy), to_np(w), mk, 64, p, np.float32)
    if act:
        t = x.double().cpu()
        ref = ref * (0.5 * (1 + torch.erf(t * 0.5 ** 0.5)) + t * torch.exp(-0.5 * t * t) * 0.3989422804014327).numpy()
    assert max_tile_rel_fro(dx, ref) <= REL_FRO_TOL
