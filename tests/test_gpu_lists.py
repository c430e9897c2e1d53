"""Kernel (a): block mask -> compacted kept-block lists, through the C ABI.  Bit-exact contract."""
import json
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import sparsedrop_oracle as O

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).parent / "golden"
CASES = json.loads((GOLDEN / "compaction_cases.json").read_text())


def _lists_np(lists):
    nnz = lists.nnz()
    return (lists.row_ptr.cpu().numpy(), lists.col_idx[:nnz].cpu().numpy(),
            lists.col_ptr.cpu().numpy(), lists.row_idx[:nnz].cpu().numpy())


@pytest.mark.parametrize("name", sorted(CASES))
def test_known_answers(name):
    from flash_dropout.hip import GEMM

    c = CASES[name]
    g = GEMM()
    mask = torch.tensor(c["mask"], dtype=torch.bool, device="cuda")
    lists = g.build_lists(mask)
    rp, ci, cp, ri = _lists_np(lists)
    assert rp.dtype == np.int32 and ci.dtype == np.int32
    assert rp.tolist() == c["row_ptr"] and ci.tolist() == c["col_idx"]
    assert cp.tolist() == c["col_ptr"] and ri.tolist() == c["row_idx"]
    table, row_indices, row_widths = g.increment_table(lists, c["block_k"])
    assert table.dtype == torch.int64
    assert table.cpu().tolist() == c["table"]
    assert row_indices.cpu().tolist() == c["row_indices"]
    assert row_widths.cpu().tolist() == c["row_widths"]


@pytest.mark.parametrize("shape,p", [((16, 16), 0.5), ((128, 128), 0.5), ((128, 128), 0.0), ((128, 128), 1.0),
                                     ((64, 13), 0.5), ((256, 6), 0.3), ((2048, 9), 0.5), ((1, 1), 0.0),
                                     ((1, 300), 0.7), ((300, 1), 0.7), ((65, 129), 0.25), ((1000, 700), 0.9)])
@pytest.mark.parametrize("col_major", [False, True])
def test_random_masks_bit_exact(shape, p, col_major):
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(shape[0] * 1000 + shape[1])
    mask_cpu = torch.rand(*shape, generator=gen) < p
    mask = mask_cpu.t().contiguous().cuda().t() if col_major else mask_cpu.cuda()
    assert tuple(mask.shape) == shape
    lists = F.kept_block_lists(mask)
    rp, ci, cp, ri = _lists_np(lists)
    erp, eci = O.compact_csr(mask_cpu.numpy())
    ecp, eri = O.compact_csc(mask_cpu.numpy())
    assert np.array_equal(rp, erp) and np.array_equal(ci, eci)
    assert np.array_equal(cp, ecp) and np.array_equal(ri, eri)
    # the library identity the reference relies on (blockwise_dropout_matmul_triton.py:48)
    nz = torch.nonzero(~mask, as_tuple=False)
    assert torch.equal(F.kept_block_table(mask), nz)
    # transposed view swaps CSR and CSC
    t = lists.transposed()
    assert t.shape == (shape[1], shape[0]) and t.row_ptr is lists.col_ptr


def test_large_mask_uses_multi_launch_path():
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(7)
    mask_cpu = torch.rand(1500, 400, generator=gen) < 0.6  # 600k entries > fused limit
    lists = F.kept_block_lists(mask_cpu.cuda())
    rp, ci, cp, ri = _lists_np(lists)
    erp, eci = O.compact_csr(mask_cpu.numpy())
    ecp, eri = O.compact_csc(mask_cpu.numpy())
    assert np.array_equal(rp, erp) and np.array_equal(ci, eci)
    assert np.array_equal(cp, ecp) and np.array_equal(ri, eri)


@pytest.mark.parametrize("shape,p,bk", [((16, 16), 0.5, 64), ((40, 70), 0.8, 128), ((9, 3), 0.95, 16)])
def test_increment_table_vs_oracle(shape, p, bk):
    import flash_dropout.functional as F

    gen = torch.Generator().manual_seed(11)
    mask_cpu = torch.rand(*shape, generator=gen) < p
    table, ri, rw = F.mask_to_increment_table(mask_cpu.cuda(), bk)
    et, eri, erw = O.mask_to_increment_table(mask_cpu.numpy(), bk)
    assert np.array_equal(table.cpu().numpy(), et)
    assert np.array_equal(ri.cpu().numpy(), eri)
    assert np.array_equal(rw.cpu().numpy(), erw)


@pytest.mark.parametrize("shape", [(1, 1), (2, 2), (5, 7), (16, 24), (63, 33), (256, 256), (600, 500)])
@pytest.mark.parametrize("p", [0.0, 0.5, 0.9])
def test_merged_lists_of_a_block_size_32_mask_bit_exact(shape, p):
    """split = 0: a mask at block size 32 listed on the 64 grid with the quadrant keep bits in bits 28-31 of every
    entry, against the oracle's encoding, for the list by rows and (transposed bits) by columns; masks larger than
    2^18 listed entries take the multi-launch builder."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    gen = torch.Generator().manual_seed(shape[0] * 1000 + shape[1])
    mask = torch.rand(*shape, generator=gen) < p
    lists = ext.build_lists(mask.cuda(), split=0)
    assert lists.shape == ((shape[0] + 1) // 2, (shape[1] + 1) // 2)
    rp, ci = O.compact_csr_quads(mask.numpy())
    assert np.array_equal(lists.row_ptr.cpu().numpy(), rp)
    assert np.array_equal(lists.col_idx[: lists.nnz()].cpu().numpy(), ci)
    cp, ri = O.compact_csr_quads(mask.numpy().T)
    assert np.array_equal(lists.col_ptr.cpu().numpy(), cp)
    assert np.array_equal(lists.row_idx[: lists.nnz()].cpu().numpy(), ri)
    # the same from a drawn mask
    drawn, lists = ext.random_lists(shape, p, seed=9, split=0)
    want = O.random_mask(shape, p, 9)
    assert np.array_equal(drawn.cpu().numpy(), want)
    rp, ci = O.compact_csr_quads(want)
    assert np.array_equal(lists.row_ptr.cpu().numpy(), rp)
    assert np.array_equal(lists.col_idx[: lists.nnz()].cpu().numpy(), ci)


@pytest.mark.parametrize("rows,cols,bs", [(96, 96, 96), (100, 130, 96), (1000, 784, 96), (4096, 4096, 160), (70, 700, 224),
                                          (8192, 8192, 96)])
@pytest.mark.parametrize("p", [0.0, 0.5, 0.9])
def test_merged_lists_of_odd_multiples_of_32_bit_exact(rows, cols, bs, p):
    """split = -k: a mask at block size 32 * k (96, 160, 224) over a [rows, cols] matrix, listed on the matrix's grid of
    64-blocks with the quadrant keep bits: against the oracle's composition (every mask entry repeated k x k times onto
    the grid of 32-blocks, that grid merged two by two), by rows and by columns, for a stored and a drawn mask."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    k = bs // 32
    shape = O.mask_shape(rows, cols, bs)
    grid64 = O.mask_shape(rows, cols, 64)
    gen = torch.Generator().manual_seed(rows + cols + bs)
    mask = torch.rand(*shape, generator=gen) < p

    def want(m):
        # the mask's 32-blocks, as far as the 64 grid reaches (a 32-block past the matrix but inside the mask's last
        # entry keeps that entry's value)
        m32 = O.split_mask(m, k, (min(shape[0] * k, 2 * grid64[0]), min(shape[1] * k, 2 * grid64[1])))
        return O.compact_csr_quads(m32), O.compact_csr_quads(m32.T)

    def check(lists, m):
        (rp, ci), (cp, ri) = want(m)
        assert lists.shape == grid64
        assert np.array_equal(lists.row_ptr.cpu().numpy(), rp)
        assert np.array_equal(lists.col_idx[: lists.nnz()].cpu().numpy(), ci)
        assert np.array_equal(lists.col_ptr.cpu().numpy(), cp)
        assert np.array_equal(lists.row_idx[: lists.nnz()].cpu().numpy(), ri)

    check(ext.build_lists(mask.cuda(), split=-k, grid=grid64), mask.numpy())
    check(ext.build_lists(mask.t().contiguous().cuda().t(), split=-k, grid=grid64), mask.numpy())  # column-major mask
    drawn, lists = ext.random_lists(shape, p, seed=11, split=-k, grid=grid64)
    assert np.array_equal(drawn.cpu().numpy(), O.random_mask(shape, p, 11))
    check(lists, O.random_mask(shape, p, 11))
    # the element mask is the one of the block size: what makes the composition the right oracle
    m32 = O.split_mask(mask.numpy(), k, O.mask_shape(rows, cols, 32))
    assert np.array_equal(O.expand_keep(m32, 32, rows, cols), O.expand_keep(mask.numpy(), bs, rows, cols))


@pytest.mark.parametrize("M,K,N,bs,merged", [
    (192, 25600, 200, 64, True),     # more entries of a workgroup's rows than it has threads, a split reduction
    (3000, 2088, 264, 96, True),     # three 32-blocks to an entry, ragged, rows of the mask that start inside a group of four
    (1056, 544, 4160, 32, True),     # 33 x 17 entries of 32-blocks
    (16400, 2048, 128, 32, True),    # 513 x 64 entries: more than the table of a list build of its own, which evaluates one by one
    (4100, 20600, 1030, 64, True),   # a full round of workgroups: a mask of 64-blocks through the table, rows of more entries than threads
    (4544, 416, 6344, 128, True),    # the same on the 256 x 256 shape or what takes its place, an entry to four blocks
    (16416, 8224, 72, 32, True),     # 513 x 257 entries: more than the table in a product's launch
])
def test_masks_evaluated_through_a_table(M, K, N, bs, merged):
    """Drawn and stored masks on both sides of the limits up to which a workgroup evaluates a mask four entries at a time into
    LDS: the mask is the oracle's, the lists are numpy's of it, and the product is the one over those lists."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    p, seed = 0.6, 91
    gen = torch.Generator("cuda").manual_seed(3)
    x = torch.randn(M, K, generator=gen, device="cuda", dtype=torch.half)
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).half()
    mask = O.random_mask(O.mask_shape(M, K, bs), p, seed)
    # keep bits of the 32-blocks of every 64-block: bit 2a + b = row half a, column half b
    mb, kb = -(-M // 64), -(-K // 64)
    fine = np.zeros((2 * mb, 2 * kb), dtype=np.int64)
    keep = np.repeat(np.repeat(~mask, bs // 32, 0), bs // 32, 1)[:2 * mb, :2 * kb]
    fine[:keep.shape[0], :keep.shape[1]] = keep
    quads = sum(fine[a::2, b::2] << (2 * a + b) for a in range(2) for b in range(2))
    rows, cols = np.nonzero(quads)
    by_col = np.lexsort((rows, cols))
    q = quads[rows, cols]
    q_t = (q & 9) | ((q & 2) << 1) | ((q & 4) >> 1)
    bits = (lambda e, b: (e | (b << 28)).astype(np.uint32).view(np.int32)) if bs % 64 else (lambda e, b: e.astype(np.int32))
    want = (np.r_[0, np.cumsum(np.bincount(rows, minlength=mb))], bits(cols, q),
            np.r_[0, np.cumsum(np.bincount(cols, minlength=kb))], bits(rows[by_col], q_t[by_col]))
    stored = torch.from_numpy(mask).cuda()
    for given in (stored, stored.t().contiguous().t(), None):
        y, m, lists, g = ext.dropout_matmul_forward(x, w, bs, p, **({"seed": seed} if given is None else {"mask": given}))
        assert ext.last_kernel_detail().startswith("dsd+lists:") == merged, ext.last_kernel_detail()
        assert np.array_equal(m.cpu().numpy(), mask)
        for a, b in zip((lists.row_ptr, lists.col_idx[:len(rows)], lists.col_ptr, lists.row_idx[:len(rows)]), want):
            assert np.array_equal(a.cpu().numpy(), b)
        alone = ext.build_lists(stored, -(bs // 32) if bs % 64 else bs // 64, (mb, kb))
        assert all(torch.equal(getattr(alone, n)[:len(b)], getattr(lists, n)[:len(b)])
                   for n, b in zip(("row_ptr", "col_idx", "col_ptr", "row_idx"), want))
        assert torch.equal(y, ext.gemm_dsd_lists(x, w, lists, g, 1 / (1 - p)))
