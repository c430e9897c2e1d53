"""CPU-side checks: the C-ABI library loads and exports what include/sparsedrop.h declares, host-side
argument validation (which runs before any GPU call), and the layer/host logic."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parent.parent


def _declared_symbols():
    text = (ROOT / "include" / "sparsedrop.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sd_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from flash_dropout.hip import _loader

    lib = _loader.load()
    declared = _declared_symbols()
    assert len(declared) >= 12
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/sparsedrop.h but not exported"
    # and the ctypes table covers exactly the header
    assert sorted(_loader.SIGNATURES) == declared
    assert lib.sd_version() >= 100


def test_workspace_bytes():
    from flash_dropout.hip import _loader

    lib = _loader.load()
    # split-K scratch: wanted for a long reduction over few tiles, not for a square problem
    assert lib.sd_splitk_workspace_bytes(576, 128, 131072, 64, 1) >= 2 * 576 * 128 * 4
    assert lib.sd_splitk_workspace_bytes(8192, 8192, 8192, 64, 1) == 0
    assert lib.sd_splitk_workspace_bytes(64, 64, 512, 64, 0) == 0
    assert lib.sd_workspace_bytes(128, 128) >= (129 + 128 * 128) * 4
    assert lib.sd_workspace_bytes(1, 1) >= 12
    assert lib.sd_workspace_bytes(-1, 4) == 0


def test_host_validation_rejects_bad_arguments_without_touching_the_gpu():
    from flash_dropout.hip import _loader

    lib = _loader.load()
    fake = ctypes.c_void_p(0x1000)
    # neither stride is 1
    rc = lib.sd_gemm(fake, 2, 2, fake, 8, 1, fake, 8, 1, 8, 8, 8, 0, None, 0, None)
    assert rc == 1 and b"row or column major" in lib.sd_last_error()
    # bad dtype
    rc = lib.sd_gemm(fake, 8, 1, fake, 8, 1, fake, 8, 1, 8, 8, 8, 7, None, 0, None)
    assert rc == 1 and b"dtype" in lib.sd_last_error()
    # row stride shorter than the row
    rc = lib.sd_gemm(fake, 4, 1, fake, 8, 1, fake, 8, 1, 8, 8, 8, 0, None, 0, None)
    assert rc == 1 and b"row stride" in lib.sd_last_error()
    # unsupported block size
    rc = lib.sd_gemm_dsd_lists(fake, 96, 1, fake, 96, 1, fake, 96, 1, fake, fake, 96, 96, 96, 48, 1.0, 0, None, 0, None)
    assert rc == 2 and b"multiples of 32" in lib.sd_last_error()
    # workspace too small
    rc = lib.sd_gemm_dsd(fake, 128, 1, fake, 128, 1, fake, 128, 1, fake, 2, 1, 128, 128, 128, 64, 2.0, 0, fake, 8, None)
    assert rc == 1 and b"workspace too small" in lib.sd_last_error()
    # null list
    rc = lib.sd_gemm_sdd_lists(fake, 128, 1, fake, 128, 1, fake, 128, 1, None, None, 128, 128, 128, 64, 2.0, 0, None)
    assert rc == 1 and b"null list" in lib.sd_last_error()
    # build_lists argument checks
    rc = lib.sd_build_lists(fake, 4, 4, 4, 1, None, None, None, None, None)
    assert rc == 1 and b"nothing to build" in lib.sd_last_error()
    rc = lib.sd_build_lists(fake, 0, 4, 4, 1, fake, fake, None, None, None)
    assert rc == 1 and b"non-empty" in lib.sd_last_error()
    # conv geometry
    rc = lib.sd_im2col(fake, 1, 1, 1, 1, fake, 4, 1, 1, 2, 2, 3, 3, 0, 0, 1, 1, 1, 1, None, None, 0, 0, None)
    assert rc == 1 and b"does not fit" in lib.sd_last_error()
    rc = lib.sd_im2col(fake, 1, 1, 1, 1, fake, 4, 1, 1, 4, 4, 3, 3, 0, 0, 1, 1, 1, 1, None, None, 0, 0, None)
    assert rc == 1 and b"cols_ld" in lib.sd_last_error()
    # the implicit-GEMM conv entry points: argument errors are reported (1), geometries without a kernel are
    # declined (2) -- both before anything is launched
    # x [1, 8, 4, 4], 3x3 without padding: P = Q = 2
    conv = [1, 8, 4, 4, 64, 3, 3, 0, 0, 1, 1, 1, 1]  # n, c, h, w, k_out, r, s, pads, strides, dilations
    rc = lib.sd_conv2d_dsd_lists(fake, 128, 16, 4, 1, fake, 72, None, 64, *conv, None, None, 64, 1.0, 0, None)
    assert rc == 1 and b"null pointer" in lib.sd_last_error()
    rc = lib.sd_conv2d_dsd_lists(fake, 128, 16, 4, 1, fake, 72, fake, 64, *conv, fake, None, 64, 1.0, 0, None)
    assert rc == 1 and b"both be given" in lib.sd_last_error()
    rc = lib.sd_conv2d_dsd_lists(fake, 128, 16, 4, 1, fake, 8, fake, 64, *conv, None, None, 64, 1.0, 0, None)
    assert rc == 1 and b"leading dimensions" in lib.sd_last_error()
    rc = lib.sd_conv2d_dsd_lists(fake, 128, 16, 4, 1, fake, 72, fake, 64, *conv, None, None, 64, 1.0, 0, None)
    assert rc == 2  # P * Q = 4 is not a multiple of 64
    rc = lib.sd_conv2d_dx(fake, 64, fake, 72, None, 128, 16, 4, 1, None, 0, 0, *conv, 64, 1.0, 0, None)
    assert rc == 1 and b"null pointer" in lib.sd_last_error()
    rc = lib.sd_conv2d_dx(fake, 64, fake, 72, fake, 128, 16, 4, 1, None, 0, 0, *conv[:9], 0, 1, 1, 1, 64, 1.0, 0, None)
    assert rc == 1 and b"strides" in lib.sd_last_error()
    rc = lib.sd_conv2d_dx(fake, 64, fake, 72, fake, 128, 16, 4, 1, fake, 1, 1, *conv, 128, 1.0, 0, None)
    assert rc == 2  # a mask at another block size than 64
    rc = lib.sd_conv2d_dw_lists(fake, 128, 16, 4, 1, fake, 64, None, 72, *conv, None, None, 64, 1.0, 0, None, 0, None)
    assert rc == 1 and b"null pointer" in lib.sd_last_error()
    assert lib.sd_conv2d_dw_workspace_bytes(128, 64, 128, 3, 3, 32, 32) >= 2 * 576 * 128 * 4
    assert lib.sd_conv2d_dw_workspace_bytes(0, 64, 128, 3, 3, 32, 32) == 0


def test_python_shim_rejects_cpu_and_fp32_operands():
    from flash_dropout.hip import GEMM

    g = GEMM()
    a = torch.randn(64, 64, dtype=torch.float16)
    with pytest.raises(ValueError, match="GPU"):
        g.gemm(a, a)
    with pytest.raises(ValueError, match="GPU"):
        g.build_lists(torch.zeros(2, 2, dtype=torch.bool))


def test_block_size_int_or_equal_pair():
    from flash_dropout.hip.binding_gemm import _block_size

    assert _block_size(64) == 64
    assert _block_size((128, 128)) == 128
    with pytest.raises(ValueError):
        _block_size((64, 128))
    with pytest.raises(ValueError):
        _block_size(0)


def test_mask_helper_matches_reference_definition():
    import flash_dropout.functional as F

    x = torch.empty(3, 784, 100)
    torch.manual_seed(5)
    m = F.blockwise_dropout_mask(x, 64, 0.5)
    torch.manual_seed(5)
    again = torch.rand(3, 13, 2) < 0.5
    assert m.dtype == torch.bool and torch.equal(m, again)
    assert not F.blockwise_dropout_mask(x, (64, 64), 0.0).any()


def test_dropout_mm_layer_host_logic():
    from flash_dropout.layers import DropoutMM

    torch.manual_seed(0)
    layer = DropoutMM(16, 8, p=0.5, variant="blockwise[naive]", block_size=4)
    assert layer.weight.shape == (8, 16) and not hasattr(layer, "bias")
    x = torch.randn(2, 3, 16)
    layer.eval()
    assert torch.allclose(layer(x), torch.nn.functional.linear(x, layer.weight))
    layer.train()
    y = layer(x)
    assert y.shape == (2, 3, 8)
    for variant in ("none", "vanilla"):
        assert DropoutMM(16, 8, variant=variant)(x).shape == (2, 3, 8)
    bad = DropoutMM(16, 8, variant="nope")
    with pytest.raises(ValueError, match="Unknown variant"):
        bad(x)
    # p = 0 block dropout is a plain linear
    l0 = DropoutMM(16, 8, p=0.0, variant="blockwise[naive]", block_size=4)
    assert torch.allclose(l0(x), torch.nn.functional.linear(x, l0.weight), atol=1e-6)


def test_naive_variant_matches_oracle_with_tails():
    import numpy as np

    import flash_dropout.functional as F
    from oracle import sparsedrop_oracle as O

    torch.manual_seed(0)
    x, w = torch.randn(10, 14, dtype=torch.float64), torch.randn(5, 14, dtype=torch.float64)
    mask = torch.rand(3, 4) < 0.5
    y = F.naive_blockwise_dropout_matmul_mask(x, mask, 4, 0.25, w)
    np.testing.assert_allclose(y.numpy(), O.dsd_forward(x.numpy(), w.numpy(), mask.numpy(), 4, 0.25), rtol=1e-12)


def test_dropout_conv_layer_host_logic():
    from flash_dropout.layers import DropoutConv2d

    torch.manual_seed(0)
    x = torch.randn(2, 3, 8, 8)
    conv = DropoutConv2d(3, 4, (3, 3), padding=(1, 1), p=0.0, variant="blockwise[naive]", block_size=4)
    ref = torch.nn.functional.conv2d(x, conv.weight, padding=(1, 1))
    assert torch.allclose(conv(x), ref, atol=1e-5)
    conv.eval()
    assert torch.allclose(conv(x), ref, atol=1e-6)
    for variant in ("none", "vanilla", "vanilla_2d"):
        assert DropoutConv2d(3, 4, (3, 3), padding=(1, 1), variant=variant)(x).shape == (2, 4, 8, 8)
    with pytest.raises(ValueError, match="Unknown variant"):
        DropoutConv2d(3, 4, (3, 3), variant="nope")(x)


@pytest.mark.parametrize("kind", [0, 1])
def test_tile_map_is_a_bijection_onto_the_tile_grid(kind):
    """The workgroup-to-tile map of the specialised kernels (the counterpart of the reference's
    threadblock_swizzle, gemm.cuh:84-97) must hit every tile of the grid exactly once, for every grid up to
    40 x 40 — totals that are not multiples of the 8 XCDs and tile-row counts that are not multiples of the
    group height included."""
    from flash_dropout.hip import _loader

    lib = _loader.load()
    tm, tn = ctypes.c_int32(), ctypes.c_int32()
    for tiles_m in range(1, 41):
        for tiles_n in range(1, 41):
            seen = set()
            for b in range(tiles_m * tiles_n):
                assert lib.sd_tile_of_block(kind, b, tiles_m, tiles_n, ctypes.byref(tm), ctypes.byref(tn)) == 0
                assert 0 <= tm.value < tiles_m and 0 <= tn.value < tiles_n, (tiles_m, tiles_n, b)
                seen.add((tm.value, tn.value))
            assert len(seen) == tiles_m * tiles_n, (tiles_m, tiles_n)
    # outside the grid: an error, not a tile
    assert lib.sd_tile_of_block(kind, 12, 3, 4, ctypes.byref(tm), ctypes.byref(tn)) == 1
    assert lib.sd_tile_of_block(2, 0, 3, 4, ctypes.byref(tm), ctypes.byref(tn)) == 1


@pytest.mark.parametrize("kind", [0, 1])
def test_group_map_is_a_bijection_for_every_number_of_sure_groups(kind):
    """What the input gradient's kernels launch by: every group that a row can have exactly once, those that are sure to exist in
    front, and with all of them sure the plain tile order."""
    from flash_dropout.hip import _loader

    lib = _loader.load()
    tm, gi, tm2, tn2 = (ctypes.c_int32() for _ in range(4))
    for rows in (1, 2, 3, 4, 5, 7, 8, 9, 17, 40):
        for groups in (1, 2, 3, 6, 7, 13):
            for sure in range(1, groups + 1):
                seen = set()
                for b in range(rows * groups):
                    assert lib.sd_group_of_block(kind, b, rows, groups, sure, ctypes.byref(tm), ctypes.byref(gi)) == 0
                    assert 0 <= tm.value < rows and 0 <= gi.value < groups
                    assert (gi.value < sure) == (b < rows * sure), (rows, groups, sure, b)
                    seen.add((tm.value, gi.value))
                    if sure == groups and kind == 1:
                        assert lib.sd_tile_of_block(1, b, rows, groups, ctypes.byref(tm2), ctypes.byref(tn2)) == 0
                        assert (tm.value, gi.value) == (tm2.value, tn2.value)
                assert len(seen) == rows * groups, (rows, groups, sure)
    for bad in ((kind, 12, 3, 4, 2), (kind, -1, 3, 4, 2), (kind, 0, 3, 4, 0), (kind, 0, 3, 4, 5), (2, 0, 3, 4, 2)):
        assert lib.sd_group_of_block(*bad, ctypes.byref(tm), ctypes.byref(gi)) == 1


def test_tile_map_keeps_an_xcd_on_a_compact_patch():
    """What the map is for: the 32 workgroups an XCD holds at a time (launch indices x, x+8, x+16, ...) cover
    at most 8 tile rows x 4+1 tile columns of a large grid, not a scattered set."""
    from flash_dropout.hip import _loader

    lib = _loader.load()
    tm, tn = ctypes.c_int32(), ctypes.c_int32()
    tiles_m = tiles_n = 32
    for x in range(8):
        rows, cols = set(), set()
        for i in range(32):
            lib.sd_tile_of_block(0, x + 8 * i, tiles_m, tiles_n, ctypes.byref(tm), ctypes.byref(tn))
            rows.add(tm.value)
            cols.add(tn.value)
        assert len(rows) <= 8 and len(cols) <= 5, (x, sorted(rows), sorted(cols))


_TAP_SWEEP = r"""
#include <stdio.h>
#include <algorithm>
#include <utility>
#include "conv_taps.h"
using namespace sd;

static long n_geometries = 0, n_small = 0, n_single = 0;

// what a launch asks for holds everything its workgroups put there
static bool lds_holds(const TapGeom& g, bool dx) {
  const int64_t span = span_of(g);
  const int64_t products = kStages * kTapStep + (span + 8) * kTapRow + (dx ? g.taps() * ((span + 63) / 64 + 2) * 17 : 4 * g.taps() * 128);
  n_small += dx && products < taps_turn_bytes(4);
  if (taps_lds(g, dx, span) < products || (dx && taps_lds(g, dx, span) < taps_turn_bytes(4))) return false;
  n_single += !dx && dw_lds(span, 2) > kLdsLimit;
  for (int buffers = 1; buffers <= 2; ++buffers)
    if (dw_lds(span, buffers) < buffers * ((span + 1) * kDwPitch + kPos * 128 + kPos * 8) || dw_lds(span, buffers) < 147456) return false;
  return true;
}

// in-image bits and windows against a loop over everything
static bool windows_hold(TapGeom g, int images) {
  g.prepare();
  const int rows = images * g.OH * g.OW, per = g.IH * g.IW;
  for (int m0 = 0; m0 < rows; m0 += kPos) {
    const int last = std::min(m0 + kPos, rows) - 1;
    const TapWindow w(g, m0, last);
    if (w.hi - w.lo > window_bound(g, kPos)) return false;
    for (int pos = m0; pos <= last; ++pos) {
      const TapPosition p(g, pos);
      if (p.img != pos / (g.OH * g.OW) || p.oh != pos % (g.OH * g.OW) / g.OW || p.ow != pos % g.OW) return false;
      uint32_t bits = 0;
      for (int t = 0; t < g.taps(); ++t) {
        const int h = p.oh - g.pad_h + t / g.S * g.dl_h, c = p.ow - g.pad_w + t % g.S * g.dl_w;
        if (h < 0 || h >= g.IH || c < 0 || c >= g.IW) continue;
        bits |= 1u << t;
        const int px = p.img * per + h * g.IW + c;
        if (px != p.pixel(g) + g.shift(t) || px < w.lo || px >= w.hi) return false;
      }
      if (bits != p.inside(g)) return false;
    }
  }
  return true;
}

static int check(int h, int w, int r, int s, int ph, int pw, int dh, int dw, bool windows) {
  const int po = h + 2 * ph - dh * (r - 1), qo = w + 2 * pw - dw * (s - 1);
  if (po < 1 || qo < 1 || r * s < 2 || r * s > 32) return 0;
  const TapGeom f{h, w, po, qo, r, s, ph, pw, dh, dw}, b{po, qo, h, w, r, s, (r - 1) * dh - ph, (s - 1) * dw - pw, dh, dw};
  if (span_of(f) > 1000 || span_of(b) > 1000) return 0;
  ++n_geometries;
  const int images = 1 + 700 / std::max(h * w, po * qo);
  if (lds_holds(f, false) && lds_holds(b, true) && (!windows || (windows_hold(f, images) && windows_hold(b, images)))) return 0;
  printf("%d x %d, kernel %d x %d, padding %d %d, dilation %d %d\n", h, w, r, s, ph, pw, dh, dw);
  return 1;
}

int main() {
  // unpadded kernels nearly as wide as the image: the gradient they read is narrow
  for (int h = 1; h <= 24; ++h)
    for (int w = 1; w <= 24; ++w)
      for (int r = 1; r <= 8; ++r)
        for (int s = 1; s <= 32; ++s)
          for (int d = 0; d < 9; ++d)
            if (check(h, w, r, s, 0, 0, 1 + d / 3, 1 + d % 3, false)) return 1;
  uint32_t x = 12345;
  auto next = [&](int lo, int hi) { x = x * 1664525u + 1013904223u; return lo + (int)((x >> 8) % (uint32_t)(hi - lo + 1)); };
  for (int i = 0; i < 6000; ++i) {
    const int r = next(1, 6), s = next(1, 6);
    if (check(next(1, 40), next(1, i % 8 ? 40 : 300), r, s, next(0, 5), next(0, 5), next(1, 3), next(1, 3), true)) return 1;
  }
  printf("%ld geometries, %ld turned in more than the products use, %ld with one buffer\n", n_geometries, n_small, n_single);
  // the layers of the device tests that are to have one buffer have it
  for (auto& l : {std::pair<int, int>{256, 3}, {160, 5}, {360, 3}}) {
    const TapGeom g{9, l.first, 9, l.first, l.second, l.second, l.second / 2, l.second / 2, 1, 1};
    if (span_of(g) < 736 || span_of(g) > 1000 || dw_lds(span_of(g), 2) <= kLdsLimit || dw_lds(span_of(g), 1) > kLdsLimit) return 1;
  }
  return n_geometries < 10000 || n_small < 100 || n_single < 10;
}
"""


def test_tap_windows_and_lds_hold_what_the_kernels_put_there(tmp_path):
    """The tap-wise convolution's geometry (csrc/conv_taps.h is plain integer code, the same on host and device): which taps lie
    inside the image, the window of source rows, its bound, and the LDS of the launches, over geometries of all kinds."""
    import subprocess

    (tmp_path / "sweep.cpp").write_text(_TAP_SWEEP)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'sparse-dropout_amd' / 'csrc'}", str(tmp_path / "sweep.cpp"), "-o",
                    str(tmp_path / "sweep")], check=True)
    proc = subprocess.run([str(tmp_path / "sweep")], capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout


@pytest.mark.parametrize("c,hw,r,stride,dil,layout,ld_off,bs,kernel", [
    (64, 32, 3, (1, 1), 1, "planes", 0, 64, "window"), (64, 32, 3, (2, 2), 1, "planes", 0, 0, "window"),
    (64, 32, 4, (2, 2), 1, "channels last", 0, 64, "window"), (64, 32, 3, (2, 2), 1, "planes", 4, 64, "elements"),
    (12, 32, 4, (2, 2), 1, "planes", 0, 64, "elements"), (64, 32, 3, (2, 2), 1, "planes", 0, 30, "elements"),
    # windows by two that fit at no height, and the widest that do
    (16, 272, 3, (2, 2), 1, "planes", 0, 64, "window"), (16, 320, 3, (2, 2), 1, "planes", 0, 64, "elements"),
    (16, 72, 5, (2, 2), 1, "planes", 0, 64, "window"), (16, 96, 5, (2, 2), 1, "planes", 0, 64, "elements"),
    (16, 32, 7, (2, 2), 1, "planes", 0, 64, "elements"), (16, 23, 7, (2, 2), 1, "planes", 0, 64, "window"),
    # other strides, dilations
    (32, 32, 3, (2, 1), 1, "planes", 0, 64, "tile"), (32, 32, 3, (1, 2), 1, "channels last", 0, 64, "tile"),
    (32, 32, 3, (2, 2), 2, "planes", 0, 64, "tile"), (32, 32, 3, (4, 4), 1, "planes", 0, 0, "tile"),
    (32, 32, 1, (1, 1), 1, "planes", 0, 64, "turn"), (12, 32, 1, (1, 1), 1, "planes", 0, 0, "turn"),
    (32, 32, 1, (1, 1), 1, "channels last", 0, 64, "window"), (32, 32, 1, (2, 2), 1, "planes", 0, 64, "window"),
    (32, 2, 5, (1, 1), 2, "planes", 0, 64, None),  # a kernel that does not fit the image
])
def test_which_kernel_folds_a_patch_gradient(c, hw, r, stride, dil, layout, ld_off, bs, kernel):
    from flash_dropout.hip import GEMM

    pad = 0 if kernel is None else dil * (r - 1) // 2 if r % 2 else 0
    strides = (hw * hw, hw, 1) if layout == "planes" else (1, hw * c, c)
    got = GEMM().lib.sd_col2im_kernel(c * r * r + ld_off, *strides, 4, c, hw, hw, r, r, pad, pad, *stride, dil, dil, bs)
    assert (None, "elements", "tile", "window", "turn")[got] == kernel


@pytest.mark.parametrize("n,c,hw,k,r,stride,dil,taken", [
    (4, 64, 32, 128, 3, 1, 1, 1), (3, 8, 32, 64, 5, 1, 1, 1), (2, 8, 32, 64, 3, 2, 1, 1), (2, 24, 32, 64, 3, 1, 2, 1),
    (2, 16, 32, 256, 1, 1, 1, 1), (2, 16, 64, 256, 1, 2, 1, 1),
    (2, 16, 64, 64, 1, 2, 1, 0),    # the open sums of 66 channels over 64-wide rows, beside half a CU's LDS
    (2, 16, 32, 64, 8, 2, 1, 1), (2, 16, 32, 64, 9, 2, 1, 0),   # 81 taps
    (2, 512, 32, 64, 3, 1, 1, 0),   # 72 block columns
    (2, 12, 32, 64, 3, 1, 1, 0),    # 108 columns
    (2, 16, 64, 64, 3, 1, 8, 0),    # taps of more output rows than the waves hold
    (2, 16, 32, 96, 3, 1, 1, 0), (2, 16, 30, 64, 3, 1, 1, 0), (2, 16, 32, 64, 3, 9, 1, 0), (0, 16, 32, 64, 3, 1, 1, 0),
])
def test_which_convolutions_have_their_input_gradient_fused(n, c, hw, k, r, stride, dil, taken):
    from flash_dropout.hip import GEMM

    lib, cols, pad = GEMM().lib, c * r * r, dil * (r - 1) // 2
    ask = lambda dy, dy_ld, w, w_ld: lib.sd_conv2d_dx_taken(dy, dy_ld, w, w_ld, n, c, hw, hw, k, r, r, pad, pad, stride, stride, dil, dil)
    assert ask(256, k, 512, cols) == taken
    assert ask(264, k, 512, cols) == ask(256, k, 520, cols) == ask(256, k + 4, 512, cols) == ask(256, k, 512, cols + 4) == 0


_RECIPROCALS = r"""
#include <stdio.h>
#include <initializer_list>
#include "reciprocal.h"

static long n_exact = 0, n_none = 0;
static bool holds(int64_t d, int64_t below) {
  const uint64_t m = sd::exact_reciprocal(d, below);
  ++(m ? n_exact : n_none);
  if (m == 0) return true;
  auto same = [&](int64_t v) { return v < 0 || v >= below || (int64_t)((uint64_t)v * m >> 32) == v / d; };
  // quotients can only be wrong next to multiples of d, and first at the largest
  for (int64_t k = 0; k <= 2000; ++k)
    if (!same(k * d - 1) || !same(k * d) || !same(((below - 1) / d - k) * d - 1) || !same((below - 1) / d * d - k * d)) return false;
  return same(below - 1);
}
int main() {
  uint64_t x = 12345;
  auto next = [&](int64_t hi) { x = x * 6364136223846793005ull + 1442695040888963407ull; return 1 + (int64_t)((x >> 20) % (uint64_t)hi); };
  for (int64_t d = 1; d <= 4096; ++d)
    for (int64_t below : {(int64_t)1, d + 100000, (int64_t)1 << 24, ((int64_t)1 << 31) + d, (int64_t)1 << 32})
      if (!holds(d, below)) return printf("%ld below %ld\n", (long)d, (long)below), 1;
  for (int i = 0; i < 20000; ++i) {
    const int64_t d = next(1LL << (1 + i % 32)), below = next(1LL << (1 + i % 33));
    if (!holds(d, below)) return printf("%ld below %ld\n", (long)d, (long)below), 1;
  }
  for (int64_t d : {(int64_t)64, (int64_t)128, (int64_t)32768, (int64_t)1 << 30})  // powers of two: for anything
    if (sd::exact_reciprocal(d, (int64_t)1 << 32) == 0) return 1;
  if (sd::exact_reciprocal(192, 20 << 20) == 0 || sd::exact_reciprocal(65535, 65540) != 0) return 1;
  return n_exact < 10000 || n_none < 1000;
}
"""


def test_reciprocals_divide_exactly_in_the_range_that_they_state(tmp_path):
    import subprocess

    (tmp_path / "sweep.cpp").write_text(_RECIPROCALS)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'sparse-dropout_amd' / 'csrc'}", str(tmp_path / "sweep.cpp"), "-o",
                    str(tmp_path / "sweep")], check=True)
    proc = subprocess.run([str(tmp_path / "sweep")], capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout


@pytest.mark.parametrize("layer,p,taken", [
    ((128, 64, 32, 32, 128, 3), 0.5, True), ((256, 32, 28, 28, 64, 3), 0.25, True), ((64, 1024, 28, 28, 128, 3), 0.75, True),
    ((64, 1024, 14, 14, 1024, 3), 0.75, False),  # 1090 us tap by tap, 649 with the dropped blocks left out
    ((8, 256, 64, 64, 256, 3), 0.95, False),     # 204, 162
    ((26, 40, 14, 14, 184, 5), 0.05, False),     # 20 workgroups, each a chain of 50 steps: 148, 98
    ((16, 16, 32, 32, 208, 5), 0.75, False),     # 134, 94
    ((97, 32, 7, 7, 144, 3), 0.25, False),       # 65, 49
])
def test_tap_by_tap_only_where_it_is_expected_to_be_faster(layer, p, taken):
    """The rule that takes a convolution to the tap-wise products knows what they cost beside the routes that skip dropped blocks."""
    from flash_dropout.hip import GEMM

    n, c, h, w, k, r = layer
    geo = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1, 1, 1)
    lib = GEMM().lib
    assert lib.sd_conv2d_taps_fits(*geo) == 1
    assert lib.sd_conv2d_taps_taken(*geo, p) == int(taken)
    assert lib.sd_conv2d_taps_taken_blocks(*geo, p, 64) == int(taken)


@pytest.mark.parametrize("layer,p,bs", [
    ((149, 80, 7, 7, 192, 3), 0.1, 64),    # 88 us without, 100 tap by tap
    ((50, 16, 30, 30, 216, 5), 0.75, 128),  # 156, 170
    ((221, 56, 7, 7, 152, 3), 0.1, 64),     # 80, 89
    ((92, 64, 14, 14, 72, 3), 0.75, 64),    # 71, 77
    ((25, 32, 30, 30, 152, 3), 0.75, 128),  # 85, 70: on the other side of the rule's error
    ((22, 40, 30, 30, 128, 3), 0.5, 64),
])
def test_how_a_weight_gradient_is_cut_moves_no_convolution_to_another_route(layer, p, bs):
    """Which route a layer takes decides how its input gradient is rounded, and the rule counts the weight gradient's parts: as many as
    fill the chip once, also in layers where fewer would take as many turns each."""
    from flash_dropout.hip import GEMM

    n, c, h, w, k, r = layer
    geo = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1, 1, 1)
    lib, rows = GEMM().lib, n * h * w
    want = max(1, 256 // (-(-c // 32) * -(-k // 64) * -(-r * r // 9)))
    parts = lib.sd_conv2d_taps_dw_workspace_bytes(c, k, r, r, rows) // (4 * r * r * c * k)
    turns = -(-rows // 256)
    assert parts == min(want, turns) and -(-turns // -(-turns // parts)) < parts
    assert lib.sd_conv2d_taps_fits(*geo) == 1 and lib.sd_conv2d_taps_taken_blocks(*geo, p, bs) == 0


def test_larger_blocks_cost_the_other_routes_more():
    """They spread such a mask over 64-blocks first: 10 x 40 x 32 x 32 -> 168 at p = 0.05 takes 94 us there in blocks of 128, 79
    tap by tap."""
    from flash_dropout.hip import GEMM

    geo = (10, 40, 32, 32, 168, 3, 3, 1, 1, 1, 1, 1, 1)
    assert [GEMM().lib.sd_conv2d_taps_taken_blocks(*geo, 0.05, bs) for bs in (64, 128)] == [0, 1]


def test_loader_refuses_a_library_built_from_other_sources(monkeypatch):
    from flash_dropout.hip import _loader

    lib = _loader.load()
    assert lib.sd_source_hash().decode() == _loader.source_hash()
    monkeypatch.setattr(_loader, "source_hash", lambda: "0" * 16)
    with pytest.raises(RuntimeError, match="built from other sources"):
        _loader.load.__wrapped__()


def test_as_matrix_lays_out_expanded_and_strided_views():
    from flash_dropout.hip.binding_gemm import _mat, as_matrix

    a = torch.zeros(6, 8)
    at = a.t()
    assert as_matrix(a) is a and as_matrix(at) is at
    assert as_matrix(a[:, :4]) is not None and as_matrix(a[:, :4]).data_ptr() == a.data_ptr()  # row stride 8 >= 4
    e = torch.zeros(1, 8).expand(6, 8)  # strides (0, 1): what y.sum(0) hands to backward
    assert as_matrix(e).stride() == (8, 1)
    assert as_matrix(a[::2, ::2]).stride() == (4, 1)
    with pytest.raises(ValueError, match="expanded view"):
        _mat(e)
    assert _mat(torch.zeros(1, 8))[1:] == (8, 1)


def test_masks_are_laid_out_before_their_strides_are_read():
    """Element (r, c) has to lie at r * strides[0] + c * strides[1] of what is launched on, expanded masks included."""
    from flash_dropout.hip.binding_gemm import _check_mask, _mask_strides

    one_row, one_col = torch.rand(1, 7) < 0.5, torch.rand(5, 1) < 0.5
    full = torch.rand(10, 14) < 0.5
    masks = [one_row.expand(5, 7), one_col.expand(5, 7), one_row[:, :1].expand(5, 7), full[:5, :7], full[:5, :7].t(),
             full[::2, ::2], one_row, one_col, one_row[:, ::2], one_row[:, :1].expand(5, 1), one_row[:, :1].expand(1, 7)]
    for mask in masks:
        m = _check_mask(mask, tuple(mask.shape), mask)
        sr, sc = _mask_strides(m)
        assert torch.equal(m, mask)
        base = m.storage_offset()
        last = base + (m.shape[0] - 1) * sr + (m.shape[1] - 1) * sc
        assert last < m.untyped_storage().nbytes()
        got = [[bool(m.untyped_storage()[base + r * sr + c * sc]) for c in range(m.shape[1])] for r in range(m.shape[0])]
        assert got == mask.tolist(), (mask.shape, mask.stride())


@pytest.mark.parametrize("name", ["mfma_ceiling.hip", "lds_load_ceiling.hip"])
def test_ceiling_probes_compile_for_gfx950(name, tmp_path):
    """The stand-alone measurement programs under benchmark/ are only ever run on a GPU box by hand: keep them
    compiling (device code for gfx950, no GPU needed)."""
    import shutil
    import subprocess

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    src = Path(__file__).resolve().parent.parent / "sparse-dropout_amd" / "benchmark" / name
    proc = subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-w", "-Xclang", "-target-feature", "-Xclang",
                           "-packed-fp32-ops", "-c", str(src), "-o", str(tmp_path / "probe.o")],
                          capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]




def test_a_traced_call_is_one_operation_on_its_tensors():
    """The recording itself, around a stand-in for the native call (its result is filled behind torch's back)."""
    from flash_dropout.functional.tracing import traceable

    class Native(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, *ws):
            ctx.save_for_backward(x, *ws)
            y = torch.empty(x.shape[0], ws[0].shape[0])
            y.numpy()[:] = sum(x.detach().numpy() @ w.detach().numpy().T for w in ws)
            return y

        @staticmethod
        def backward(ctx, g):
            x, *ws = ctx.saved_tensors
            return (sum(g @ w for w in ws), *(g.t() @ x for _ in ws))

    @traceable
    def product(x, ws, flag, mask=None):
        assert flag == "flag" and (mask is None or mask.dtype == torch.bool)
        return Native.apply(x if mask is None else x * mask, *ws)

    def f(x, a, b, mask):
        return product(x, (w for w in (a, b)), "flag", mask=mask) * 2

    make = lambda seed: [torch.randn(*s, generator=torch.Generator().manual_seed(seed)).requires_grad_()  # noqa: E731
                         for s in ((5, 4), (3, 4), (3, 4))] + [torch.arange(4) % 2 == seed % 2]
    traced = torch.jit.trace(f, tuple(make(0)), check_trace=False)
    args = make(1)
    got, want = traced(*args), f(*args)
    assert torch.equal(got, want)
    dy = torch.randn(5, 3)
    assert all(torch.equal(s, t) for s, t in zip(torch.autograd.grad(got, args[:3], dy), torch.autograd.grad(want, args[:3], dy)))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(got, args[:3], dy)


def test_the_generator_is_asked_only_where_a_mask_is_drawn(monkeypatch):
    import sys

    import flash_dropout.functional as F

    mod = sys.modules[F.hip_blockwise_dropout_mlp.__module__]
    calls = []
    monkeypatch.setattr(mod, "draw_source", lambda like, seed: calls.append(seed) or (None, "state"))
    monkeypatch.setattr(mod._loader, "bridge", lambda: type("B", (), {"mlp": staticmethod(lambda *a: a)}))
    x, w, m = torch.zeros(4, 4), [torch.zeros(4, 4)] * 2, torch.zeros(1, 1, dtype=torch.bool)
    for args, kw, drawn in (((w, 64, 0.5), dict(masks=[m, m]), False), ((w, 64, 0.5), dict(masks=[m, None]), True),
                            ((w, 64, 0.5), {}, True), ((w[:1], 64, 0.0), {}, False), ((w[:1], 64, 0.1), {}, True)):
        calls.clear()
        out = F.hip_blockwise_dropout_mlp(x, *args, **kw)
        assert bool(calls) == drawn and out[-1] == ("state" if drawn else None)
    assert F.hip_blockwise_dropout_mlp(x.requires_grad_(), w[:1], 64, 0.0)[-1] == "state"  # draws the (all kept) mask


@pytest.mark.parametrize("geometry", [dict(stride=0), dict(stride=(1, -1)), dict(dilation=0), dict(padding=(0, -1))])
def test_conv_geometry_is_checked_before_it_is_used(geometry):
    """(also in front of every other check of the operands: a stride of 0 is a division by zero in native code)"""
    import flash_dropout.functional as F

    x, k = torch.zeros(1, 4, 8, 8, dtype=torch.float16), torch.zeros(4, 4, 3, 3, dtype=torch.float16)
    for call in (lambda: F.im2col_conv2d(x, k, **geometry),
                 lambda: F.blockwise_dropout_conv2d_mask(x, torch.zeros(1, 1, dtype=torch.bool), 64, 0.5, k, **geometry)):
        with pytest.raises(ValueError, match="strides and dilations"):
            call()
