"""fp16 convolution on weights in the reference's blocked layout (csrc/conv_direct.hpp, transpose8): the sizes between which its
planner changes tiles, and half a channel tile at the end, against sums of small integers that fp32 holds exactly."""
import pytest
import torch

import unit_amd as U

pytestmark = pytest.mark.gpu

# N, C, H, W, K, window, stride, tile
SHAPES = [
    (1, 16, 7, 7, 16, 1, 1, None),                   # one k-step, one channel block
    (4, 32, 20, 26, 608, 3, 1, "x64_y32_g4_d6"),     # 270 tiles of 64 x 64, 18 k-steps
    (1, 176, 74, 61, 208, 3, 1, "x64_y128_g4_d3"),   # 268 tiles, long
    (3, 80, 65, 39, 240, 3, 1, "x64_y128_g4_d3"),    # 440 tiles
    (1, 112, 70, 66, 496, 3, 1, "x64_y64_g2_d6"),    # more than 512 tiles, half a tile of channels at the end
    (15, 160, 14, 20, 1008, 3, 1, "x64_y128_g4_d3"), # 816 tiles, 90 k-steps
    (7, 64, 36, 44, 336, 3, 1, "x64_y64_g1_d4"),     # 36 k-steps
    (7, 80, 37, 41, 352, 3, 1, "x64_y64_g1_d6"),     # 45 k-steps
    (6, 80, 46, 66, 400, 3, 1, "x64_y64_g1_d4"),     # more than 1568 tiles
    (2, 48, 31, 33, 272, 5, 2, None),
    (12, 80, 62, 50, 32, 3, 1, "x32_y64_g4_d6n"),     # 32 channels, 45 k-steps
    (8, 48, 70, 66, 16, 3, 1, "x32_y64_g4_d6n"),     # 16 channels, 27 k-steps
    (13, 80, 26, 22, 1264, 3, 2, "x64_y64_g2_d6n"),  # 500 tiles, 260 of 64 x 128
    (11, 96, 16, 15, 1904, 3, 1, "x64_y64_g1_d6n"),  # 960 tiles, 54 k-steps: below the next line
    (13, 96, 16, 15, 1904, 3, 1, "x64_y64_g1_d6hn"), # 1110 tiles, 54 k-steps: eight loads per fragment
    (14, 96, 17, 15, 1744, 3, 1, "x64_y64_g1_d6hn"), # 1204 tiles, half a tile of channels at the end
    (20, 96, 40, 33, 144, 3, 1, "x64_y64_g1_d6hn"),
    (45, 64, 18, 17, 912, 1, 1, "x64_y64_g1_d3w4n"), # 3240 tiles, four k-steps
    (9, 32, 70, 70, 688, 1, 1, "x64_y64_g1_d6n"),    # 7590 tiles, two k-steps
    (12, 32, 80, 60, 1648, 3, 2, "x64_y64_g1_d4n"),  # 5538 tiles, 18 k-steps
    (12, 32, 80, 112, 1648, 3, 2, "x64_y64_g1_d3n"), # 10478 tiles
    (16, 512, 7, 7, 2048, 1, 1, "x64_y128_g4_d3n_r4"),  # table rows
    (256, 1024, 14, 14, 512, 1, 2, "x128_y64_g1_d3n"),
]


@pytest.mark.parametrize("N,C,H,W,K,k,s,tile", SHAPES)
def test_against_float(N, C, H, W, K, k, s, tile):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N + C + K)
    x = torch.randint(-4, 5, (N, C, H, W), device=dev, generator=g).half()
    w = torch.randint(-3, 4, (K, C, k, k), device=dev, generator=g).half()
    blocked = U.prepack_conv_weight_f16(w)
    xb = U.pack_nchwc(x, 16)
    out = U.conv2d_NCHW16c_OHWI16o(xb, blocked, s, s)
    assert U.last_variant().startswith("f16direct_" + (tile or "")), U.last_variant()
    oh, ow = (H - k) // s + 1, (W - k) // s + 1
    ref = torch.zeros((N, oh, ow, K), device=dev)  # integers below 2^24: exact
    xs = x.float().permute(0, 2, 3, 1).contiguous()
    for kh in range(k):
        for kw in range(k):
            rows = xs[:, kh:kh + (oh - 1) * s + 1:s, kw:kw + (ow - 1) * s + 1:s].reshape(-1, C)
            ref += torch.mm(rows, w[:, :, kh, kw].float().t().contiguous()).view_as(ref)
    assert torch.equal(out.permute(0, 2, 3, 1, 4).reshape(N, oh, ow, K), ref)
