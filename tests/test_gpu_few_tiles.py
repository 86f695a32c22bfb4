"""Convolutions with a long reduction and few output pixels: tiles of one 32-channel block whose k-steps eight waves share.
Odd tap counts, channel counts that leave half a block, pixels that end inside a tile, fewer k-steps than the waves'
rings hold, and both sides of the rule's limits (20 k-steps, in fp16 25, 256 tiles of 32 x 32, 32 channels)."""
import numpy as np
import pytest
import torch

import unit_amd as U

pytestmark = pytest.mark.gpu

# N, C, H, W, K, window, stride, pad; the tile the rule takes
SHAPES = [(1, 640, 4, 5, 16, 1, 1, 0, "x32_y32_g8"), (2, 80, 6, 7, 48, 3, 2, 1, "x32_y32_g8"),
          (3, 336, 9, 7, 80, 3, 1, 1, "x32_y32_g8"), (1, 48, 12, 11, 32, 5, 1, 0, "x32_y32_g8"),
          (8, 80, 32, 32, 32, 3, 1, 1, "x32_y32_g8"), (8, 80, 33, 33, 32, 3, 1, 1, "x32_y64_g8"),
          (8, 80, 33, 33, 48, 3, 1, 1, "x64_y"), (2, 624, 6, 7, 48, 1, 1, 0, "x64_y32_g4")]


@pytest.mark.parametrize("N,C,H,W,K,ks,stride,pad,tile", SHAPES)
def test_int8(dev, oracle, N, C, H, W, K, ks, stride, pad, tile):
    g = np.random.RandomState(C + K)
    x = g.randint(0, 256, (N, C // 16, H, W, 16)).astype(np.uint8)
    w = g.randint(-128, 128, (K // 16, C // 16, ks, ks, 4, 16, 4)).astype(np.int8)
    ref = oracle.c_conv2d_nchwc(x, w, stride, pad, 1)
    t = lambda a: torch.from_numpy(a).to(dev)
    for weight in (t(w), U.prepare_conv2d_weight(t(w))):
        out = U.conv2d_NCHWc_int8(t(x), weight, stride, pad).cpu().numpy()
        name = U.last_variant()
        assert np.array_equal(out, ref), name
        assert tile in name, name
        # signed data x - 128: the oracle's sums less 128 sum(w), which the same operator gives on a constant
        shift = oracle.c_conv2d_nchwc(np.full_like(x, 128), w, stride, 0, 1) if pad == 0 else None
        if shift is not None:
            s8 = t((x.astype(np.int16) - 128).astype(np.int8))
            fused = U.conv2d_NCHWc_int8_fused(s8, weight, torch.zeros(K, dtype=torch.int32, device=dev), 1, stride, pad)
            assert np.array_equal(fused.cpu().numpy(), ref - shift), U.last_variant()


@pytest.mark.parametrize("N,C,H,W,K,ks,stride", [(1, 320, 4, 5, 16, 1, 1), (2, 48, 7, 6, 48, 3, 2), (3, 176, 9, 8, 80, 3, 1),
                                                 (1, 16, 12, 11, 32, 5, 1), (8, 48, 34, 35, 32, 3, 1)])
def test_fp16(dev, oracle, N, C, H, W, K, ks, stride):
    g = np.random.RandomState(C + K)
    a = g.randint(-3, 4, (N, C // 16, H, W, 16)).astype(np.float16)  # integers: exact in any order
    b = g.randint(-2, 3, (K // 16, C // 16, ks, ks, 16, 16)).astype(np.float16)
    ref = oracle.conv2d_nchw16c_f16(a, b, stride, stride)
    t = lambda v: torch.from_numpy(v).to(dev)
    for weight in (t(b), U.prepare_conv2d_weight(t(b))):
        out = U.conv2d_NCHW16c_OHWI16o(t(a), weight, stride, stride).cpu().numpy()
        assert np.array_equal(out.astype(np.float64), ref) and "_g8_" in U.last_variant(), U.last_variant()


@pytest.mark.parametrize("C,K,stride,tile", [(384, 48, 1, "x64_y32_g4"), (352, 560, 2, "x64_y32_g4"), (400, 48, 1, "x32_y32_g8"),
                                             (320, 16, 2, "x64_y32_g4"), (384, 16, 1, "x32_y32_g8")])
def test_fp16_short_reductions(dev, oracle, C, K, stride, tile):
    """Up to 24 k-steps the four waves of the wider tiles hold the whole reduction in flight."""
    g = np.random.RandomState(C + K)
    a = g.randint(-3, 4, (1, C // 16, 16, 33, 16)).astype(np.float16)
    b = g.randint(-2, 3, (K // 16, C // 16, 1, 1, 16, 16)).astype(np.float16)
    ref = oracle.conv2d_nchw16c_f16(a, b, stride, stride)
    t = lambda v: torch.from_numpy(v).to(dev)
    for weight in (t(b), U.prepare_conv2d_weight(t(b))):
        out = U.conv2d_NCHW16c_OHWI16o(t(a), weight, stride, stride).cpu().numpy()
        assert np.array_equal(out.astype(np.float64), ref) and tile in U.last_variant(), U.last_variant()


@pytest.mark.parametrize("C,H,W,K,KH,KW,tile", [
    (60, 9, 8, 48, 5, 5, "x32_y32_g8"),    # 75 window rows
    (1056, 38, 8, 32, 31, 1, "x64_y32_g4"),  # 8184 rows: their table leaves no room for the eight waves' tiles
    (524, 38, 8, 32, 31, 1, "x32_y32_g8"),   # 4061 rows
])
def test_four_channel_blocks(dev, oracle, C, H, W, K, KH, KW, tile):
    g = np.random.RandomState(C + K)
    x = g.randint(0, 256, (1, C // 4, H, W, 4)).astype(np.uint8)
    w = g.randint(-128, 128, (K // 16, C // 4, KH, KW, 1, 16, 4)).astype(np.int8)
    ref = oracle.c_conv2d_nchwc(x, w, 1, 0, 1)
    signed = oracle.conv2d_nchwc_int8_fused(x.view(np.int8), w, np.zeros(K, np.int32), 1, 1, 0, 1, conv=oracle.c_conv2d_nchwc)
    t = lambda a: torch.from_numpy(a).to(dev)
    for weight in (t(w), U.prepare_conv2d_weight(t(w))):
        out = U.conv2d_NCHWc_int8(t(x), weight, 1, 0)
        assert np.array_equal(out.cpu().numpy(), ref) and tile in U.last_variant(), U.last_variant()
        fused = U.conv2d_NCHWc_int8_fused(t(x.view(np.int8)), weight, None, 1, 1, 0)
        assert np.array_equal(fused.cpu().numpy(), signed) and tile in U.last_variant(), U.last_variant()
