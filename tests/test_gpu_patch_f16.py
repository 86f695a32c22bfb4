"""The fp16 3 x 3 convolution with pixels through LDS (conv_patch_f16.hip) against float64: tiles that begin and end inside rows and
images, patches over several images, channel blocks that do not divide among the waves, channels past the last tile."""
import pytest
import torch

import unit_amd as U

pytestmark = pytest.mark.gpu

# N, C, H, W, K; patch size in pixels
SHAPES = [(32, 256, 16, 16, 256, 256), (38, 304, 13, 17, 272, 256), (260, 320, 6, 5, 560, 384), (9, 368, 30, 28, 224, 384),
          (8, 368, 30, 28, 240, 384), (8, 272, 58, 58, 64, 512), (1, 336, 88, 88, 240, 512), (1, 512, 62, 86, 304, 512)]


@pytest.mark.parametrize("N,C,H,W,K,patch", SHAPES)
def test_against_float64(dev, N, C, H, W, K, patch):
    g = torch.Generator(device=dev).manual_seed(N + C + K)
    # small integers: exact in fp32 sums of any order
    x = torch.randint(-4, 5, (N, C, H, W), device=dev, generator=g).half()
    w = torch.randint(-3, 4, (K, C, 3, 3), device=dev, generator=g).half()
    prepared = U.prepare_conv2d_weight(U.prepack_conv_weight_f16(w))
    out = U.conv2d_NCHW16c_OHWI16o(U.pack_nchwc(x, 16), prepared, 1, 1)
    assert U.last_variant() == f"f16prep_patch_x64_y128_g4_p{patch}", U.last_variant()
    ref = torch.zeros((N, H - 2, W - 2, K), device=dev, dtype=torch.float32)  # integers below 2^24: exact
    xs = x.float().permute(0, 2, 3, 1).contiguous()
    for kh in range(3):
        for kw in range(3):
            ref += torch.mm(xs[:, kh:kh + H - 2, kw:kw + W - 2].reshape(-1, C), w[:, :, kh, kw].float().t().contiguous()).view_as(ref)
    got = out.permute(0, 2, 3, 1, 4).reshape(N, H - 2, W - 2, K)
    assert torch.equal(got, ref)


def test_infinities_stay_in_their_windows(dev):
    """A pixel past the last one, or past an image, must not reach a sum."""
    x = torch.ones((32, 256, 16, 16), device=dev, dtype=torch.float16)
    x[5, 7, 3, 9] = float("inf")
    w = U.prepare_conv2d_weight(U.prepack_conv_weight_f16(torch.ones((256, 256, 3, 3), device=dev, dtype=torch.float16)))
    out = U.conv2d_NCHW16c_OHWI16o(U.pack_nchwc(x, 16), w, 1, 1)
    assert U.last_variant().startswith("f16prep_patch_")
    bad = torch.isinf(out).nonzero()
    assert len(bad) == 9 * 256 and set(map(tuple, bad[:, [0, 2, 3]].tolist())) == {(5, h, v) for h in (1, 2, 3) for v in (7, 8, 9)}
    assert torch.equal(out[~torch.isinf(out)], torch.full_like(out[~torch.isinf(out)], 2304.0))


# N, C, H, W, K where other kernels are faster: a measured choice of the table, 128-channel tiles that fill the chip, a second round
# that few channel blocks do not pay for, one round of short reductions
OTHERS = [(256, 512, 9, 9, 512, "f16lds_"), (20, 336, 25, 33, 512, "f16prep_x128_y64_"), (9, 288, 18, 20, 1456, "f16prep_x64_y64_"),
          (102, 144, 16, 21, 48, "f16prep_x64_y64_"), (6, 832, 49, 73, 96, "f16prep_x64_y64_")]


@pytest.mark.parametrize("N,C,H,W,K,name", OTHERS)
def test_shapes_that_stay_with_other_kernels(dev, N, C, H, W, K, name):
    w = U.prepare_conv2d_weight(torch.ones((K // 16, C // 16, 3, 3, 16, 16), device=dev, dtype=torch.float16))
    out = U.conv2d_NCHW16c_OHWI16o(torch.ones((N, C // 16, H, W, 16), device=dev, dtype=torch.float16), w, 1, 1)
    assert U.last_variant().startswith(name), U.last_variant()
    assert (out == 9.0 * C).all()


@pytest.mark.parametrize("pin", ["UNIT_AMD_CONV_VARIANT", "UNIT_AMD_CONV_PANEL", "UNIT_AMD_CONV_SPLITK"])
def test_pinned_plans_reach_the_other_kernels(dev, monkeypatch, pin):
    N, C, H, W, K, _ = SHAPES[0]
    w = U.prepare_conv2d_weight(torch.ones((K // 16, C // 16, 3, 3, 16, 16), device=dev, dtype=torch.float16))
    x = torch.ones((N, C // 16, H, W, 16), device=dev, dtype=torch.float16)
    monkeypatch.setenv(pin, "60" if pin.endswith("VARIANT") else "1")
    out = U.conv2d_NCHW16c_OHWI16o(x, w, 1, 1)
    assert "patch" not in U.last_variant(), U.last_variant()
    assert (out == 9.0 * C).all()
