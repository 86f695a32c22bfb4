"""The chain kernel's wave tiles (64 x 64, 64 x 32, 32 x 32 channels x pixels) with every k-group count and tap walk, channels and pixels
that end inside a tile, a last group of fewer images; bit-exact against the oracle's operators chained the same way."""
import numpy as np
import pytest

from test_gpu_chain import _oracle_chain, _t, _to_chain
from test_gpu_chain_kernel import _build
from unit_amd import chain, rng

pytestmark = pytest.mark.gpu

# (oc, (kh, kw), stride, padding, source or None for the layer before), images, channels, rows, columns
CASES = {
    "large": ([(64, (3, 3), 1, 1, None), (80, (1, 1), 1, 0, None), (272, (1, 1), 1, 0, None), (64, (3, 3), 1, 0, None),
               (208, (3, 3), 1, 1, 0), (64, (2, 3), 1, (1, 1, 0, 1), 0), (336, (1, 1), 1, 0, 0), (48, (5, 5), 1, 2, 0),
               (96, (1, 1), 1, 0, 6), (128, (3, 3), 1, 1, 0), (16, (1, 1), 1, 0, None)], 11, 64, 41, 37),
    "half": ([(128, (3, 3), 1, 1, None), (144, (1, 1), 1, 0, None), (128, (3, 2), 1, 0, 0), (112, (3, 3), 1, 1, 0),
              (304, (1, 1), 1, 0, 0), (176, (1, 1), 2, 0, 0), (96, (1, 3), 1, (0, 1, 0, 1), 0), (144, (3, 3), 2, 1, 0),
              (128, (1, 1), 1, 0, 0), (560, (1, 1), 1, 0, 0), (64, (1, 1), 1, 0, 9)], 7, 128, 28, 27),
}


@pytest.mark.parametrize("name", CASES)
def test_tiles_bit_exact(dev, oracle, name):
    spec, n, c0, h, w = CASES[name]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    for o in c.outputs:
        o.fill_(77)
    c(_t(x, dev))
    for i, (got, ref) in enumerate(zip(c.outputs, want)):
        assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({c.variants[i]})"
    # k-steps in flight: 64 x 64, 64 x 32, 32 x 32
    assert {v.split("_")[4] for v in c.variants} == {"d5", "d6", "d9"}, c.variants


@pytest.mark.parametrize("hw", [7, 30])
def test_scales_too_wide_to_double(dev, oracle, hw):
    """Scales from 2^30 on leave the shift below 33: the 64-bit form of the requantisation, on whole blocks and on quarters."""
    x = rng.uniform_u8((3, 4, hw, hw, 16), 5)
    layers = []
    for i, (oc, k) in enumerate([(64, 1), (64, 3), (32, 1), (256, 3), (512, 1), (64, 1), (64, 3), (64, 1), (64, 1), (64, 1), (64, 1)]):
        ic = layers[-1][0].shape[0] if layers else 64
        wt = (rng.uniform_s8((oc, ic, k, k), 30 + i) % 3 - 1).astype(np.int8)
        layers.append((wt, None, (1 << 30) + 12345 * i, 32 - i % 3, 1, k // 2, i - 1))
    want = _oracle_chain(oracle, layers, x)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    c(_t(x, dev))
    for i, (got, ref) in enumerate(zip(c.outputs, want)):
        assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({c.variants[i]})"
    assert all(v.startswith("q8chain_") for v in c.variants), c.variants
    assert 0.01 < (want[-1] > 0).mean() and len(np.unique(want[-1])) > 16


# 3 x 3 windows over a patch of pixels in LDS: rows of a patch that end on a load of 64 pixels or one past it (32 + 2 W + 2 and
# 64 + 2 W + 2 pixels), images of a row or a column, tiles over many images; 96 channels have no whole periods of nine k-steps
@pytest.mark.parametrize("n,c,h,w", [(1, 128, 14, 14), (2, 128, 9, 15), (9, 128, 1, 5), (3, 128, 6, 1), (33, 128, 7, 7), (17, 64, 31, 30), (24, 128, 30, 30),
                                     (24, 128, 29, 31), (1, 128, 20, 47), (5, 512, 7, 7), (8, 512, 5, 20), (16, 512, 5, 31), (3, 96, 17, 12)])
def test_patches_bit_exact(dev, oracle, n, c, h, w):
    spec = [(c, (3, 3), 1, 1, None)] * (3 if c >= 512 else 10) + [(32, (1, 1), 1, 0, None)] * (8 if c >= 512 else 1)
    x, layers, want = _build(oracle, spec, n, c, h, w)
    ch = chain.ConvChain(_to_chain(layers, dev), x.shape)
    for _ in range(2):
        for o in ch.outputs:
            o.fill_(77)
        ch(_t(x, dev))
        for i, (got, ref) in enumerate(zip(ch.outputs, want)):
            assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({ch.variants[i]})"
    assert all(v.startswith("q8chain_") for v in ch.variants), ch.variants
    walks = {v.split("_")[5] for v, (oc, *_) in zip(ch.variants, spec) if oc == c}
    assert walks == ({"m2"} if c == 96 else {"m4"}), ch.variants


@pytest.mark.parametrize("w,walk", [(46, "m4"), (47, "m3")])
def test_largest_patch(dev, oracle, w, walk):
    """512 channels in four k-groups: 8 channel blocks of 2 rows of 64 pixels fill a wave's 16 KiB, with 47 columns there are 3 rows."""
    spec = [(64, (3, 3), 1, 1, -1)] + [(16, (1, 1), 1, 0, None)] * 8
    x, layers, want = _build(oracle, spec, 9, 512, 2, w)
    ch = chain.ConvChain(_to_chain(layers, dev), x.shape)
    ch(_t(x, dev))
    assert [v.split("_")[3:6] for v in ch.variants[:1]] == [["g4", "d9", walk]], ch.variants
    for i, (got, ref) in enumerate(zip(ch.outputs, want)):
        assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({ch.variants[i]})"


ONES = [(16, (1, 1), 2, 0, -1)] + [(16, (1, 1), 1, 0, None)] * 10  # so that the chain is long enough for the kernel
UNEVEN = (2, 0, 1, 1)
# layers that each read the chain's input; images, channels, rows, columns; what they are there for: k-steps in flight of the general
# walk (5, 6, 9: tiles of 64 x 64, 64 x 32, 32 x 32), k-groups, walk (0 one tap, 1 without padding, 2 any window, 3 whole periods of 3 x 3
# windows, 4 the same from a patch in LDS)
WALKS = {
    "16_channels": ([(512, (5, 5), 1, 2, -1), (1024, (1, 1), 1, 0, -1), (400, (1, 1), 1, 0, -1), (400, (1, 3), 1, (0, 1, 0, 1), -1),
                     (1024, (1, 3), 1, (0, 1, 0, 1), -1), (400, (3, 3), 1, 0, -1), (208, (3, 3), 1, 0, -1), (208, (3, 3), 1, UNEVEN, -1),
                     (208, (5, 5), 1, 2, -1)], 9, 16, 20, 15, "522 511 611 612 512 621 641 622 542"),
    "32_channels": ([(80, (1, 1), 1, 0, -1), (80, (3, 3), 1, 0, -1), (48, (1, 1), 1, 0, -1), (48, (3, 3), 1, 0, -1), (80, (3, 3), 1, 1, -1),
                     (48, (3, 3), 1, 1, -1), (80, (5, 5), 2, 0, -1), (48, (2, 3), 1, 0, -1)], 9, 32, 56, 51,
                    "510 513 610 613 514 614 541 521"),
    "small_images": ([(512, (3, 1), 1, 0, -1), (208, (1, 3), 1, (0, 1, 0, 1), -1), (16, (3, 3), 1, 1, -1), (16, (3, 1), 1, 0, -1),
                      (16, (2, 3), 1, 0, -1), (16, (1, 3), 1, (0, 1, 0, 1), -1), (16, (3, 3), 2, 1, -1), (16, (1, 1), 2, 0, -1),
                      (512, (3, 3), 1, 2, -1)], 9, 32, 7, 3, "911 912 914 921 941 922 942 910 913"),
    "64_channels_small_images": ([(1024, (1, 3), 1, (0, 1, 0, 1), -1), (16, (3, 3), 1, 2, -1), (16, (3, 3), 1, 1, -1)] + ONES[:5], 11, 64, 7, 5,
                                 "642 923 924"),
    "64_channels": ([(400, (3, 3), 1, UNEVEN, -1), (208, (3, 3), 1, UNEVEN, -1), (208, (3, 3), 1, 1, -1)] + ONES, 9, 64, 20, 15, "523 623 624"),
    "64_channels_large_images": ([(80, (3, 3), 1, 1, -1)] + ONES, 9, 64, 41, 38, "524"),
    "128_channels": ([(512, (3, 3), 1, 1, -1), (16, (1, 1), 2, 0, -1), (16, (3, 3), 2, 1, -1), (1024, (1, 1), 1, 0, -1),
                      (1024, (3, 3), 1, UNEVEN, -1), (512, (1, 1), 1, 0, -1), (512, (3, 3), 1, UNEVEN, -1), (16, (3, 3), 1, 1, -1)], 9, 128, 10, 8,
                     "644 940 943 620 543 640 643 944"),
    "256_channels": ([(48, (3, 3), 1, 1, -1), (80, (1, 1), 1, 0, -1), (16, (1, 1), 1, 0, -1)] + ONES, 9, 256, 41, 37, "544 520 920"),
    "512_channels": ([(80, (1, 1), 1, 0, -1)] + ONES, 9, 512, 28, 23, "540"),
}


def test_walks_are_all_listed():
    listed = [kind for *_, kinds in WALKS.values() for kind in kinds.split()]
    assert sorted(listed) == sorted(d + g + m for d in "569" for g in "124" for m in "01234")


@pytest.mark.parametrize("name", WALKS)
def test_every_walk_on_every_tile_bit_exact(dev, oracle, name):
    spec, n, c0, h, w, kinds = WALKS[name]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    for _ in range(2):
        for o in c.outputs:
            o.fill_(77)
        c(_t(x, dev))
        for i, (got, ref) in enumerate(zip(c.outputs, want)):
            assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({c.variants[i]})"
    for kind, v in zip(kinds.split(), c.variants):
        d, g, m = kind
        ring = {"53": 3, "54": 3, "63": 3, "64": 9}.get(d + m, int(d))
        if m == "0" and int(v.split("_r")[1]) != ring:  # a wave's whole share
            ring = 2 if d == "5" else 4
        assert v.split("_", 3)[3] == f"g{g}_d{d}_m{m}_r{ring}", (kind, v)
