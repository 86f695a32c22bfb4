"""Which chains run as one persistent kernel: the library's answer (unit_conv_chain_u8_ws_bytes) for chains that were timed both
ways.  Addresses only, nothing is launched."""
import ctypes

import pytest

from unit_amd import _lib, chain
from unit_amd._lib import ChainLayerDesc, ConvDesc


def _workspace(specs, n, c0, h, w):
    """specs: (oc, window, stride, source or None for the layer before); padding window // 2"""
    L = _lib.load()
    layers, shapes = (ChainLayerDesc * len(specs))(), []
    for i, (oc, k, stride, source) in enumerate(specs):
        source = i - 1 if source is None else source
        c, hh, ww = (c0, h, w) if source < 0 else shapes[source]
        d = ConvDesc(n, c, hh, ww, oc, k, k, stride, stride, *[k // 2] * 4, 1, 1, 16)
        oh, ow = ctypes.c_int32(), ctypes.c_int32()
        _lib.check(L.unit_conv_out_hw(ctypes.byref(d), ctypes.byref(oh), ctypes.byref(ow)))
        shapes.append((oc, oh.value, ow.value))
        y = layers[i]
        y.desc, y.prepared, y.out, y.scale, y.shift = d, (1 << 40) + (i << 30), (1 << 50) + (i << 34), 3, 14
        y.data = None if source < 0 else layers[source].out
    size = ctypes.c_size_t()
    _lib.check(L.unit_conv_chain_u8_ws_bytes(layers, len(specs), ctypes.byref(size)))
    return size.value


class _Shape:
    def __init__(self, *shape):
        self.shape = shape


def _net(make):
    return [(ly.weight.shape[0], ly.weight.shape[2], ly.stride, ly.source) for ly in make(lambda oc, ic, k: _Shape(oc, ic, k, k))]


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 16, 17, 32, 64, 128])
def test_networks_take_the_kernel(n):
    for make in (chain.resnet18_layers, chain.resnet50_layers):
        assert _workspace(_net(make), n, 64, 56, 56) > 0


# (specs, N, C, H, W), measured: microseconds in the kernel / as launches
LAUNCHES = {
    "wide images, 53.0 / 44.5": ([(32, 1, 1, None)] * 6, 61, 128, 63, 63),
    "two images, 42.9 / 38.0": ([(528, 1, 1, None), (96, 1, 1, None), (688, 3, 1, None), (64, 3, 1, None), (48, 1, 2, None),
                                 (208, 1, 1, None), (48, 1, 1, None), (16, 1, 1, None), (112, 1, 1, None)], 2, 224, 20, 20),
    "two images, deep layers, 45.4 / 39.6": ([(176, 3, 2, None), (48, 3, 1, None), (608, 1, 1, None), (80, 3, 1, None), (128, 1, 1, None),
                                              (432, 1, 1, None), (624, 3, 1, None), (464, 1, 1, None), (32, 1, 1, None)], 2, 32, 24, 24),
    "two layers, 13.7 / 7.9": ([(64, 3, 1, None)] * 2, 1, 64, 56, 56),
    "one layer": ([(64, 3, 1, None)], 32, 64, 56, 56),
}


@pytest.mark.parametrize("name", LAUNCHES)
def test_chains_that_lose_in_the_kernel_stay_launches(name):
    assert _workspace(*LAUNCHES[name]) == 0


# The estimate with the tiles taken, where 64 x 64 alone (and k-groups that leave whole periods or not) said launches
KERNEL = {
    "six images of 8 x 8, 19.9 / 27.2": ([(48, 3, 1, None)] * 3 + [(192, 3, 1, None)] * 3, 6, 48, 8, 8),
    "narrow layers, 23.1 / 29.9": ([(16, 3, 1, None), (80, 3, 1, None), (96, 3, 1, None), (16, 3, 1, None), (16, 1, 1, None),
                                    (48, 3, 1, None), (96, 3, 1, None)], 6, 272, 7, 7),
    "24 images, 40.1 / 49.9": ([(32, 3, 1, None)] * 4 + [(336, 3, 1, None), (304, 3, 1, None)], 24, 32, 28, 21),
}


@pytest.mark.parametrize("name", KERNEL)
def test_chains_that_win_with_small_tiles_take_the_kernel(name):
    assert _workspace(*KERNEL[name]) > 0
