"""Chains that run as one persistent kernel, bit-exact against the oracle's operators chained the same way: tiles with
idle waves, one, two and four k-groups, groups of images of which the last one is smaller, flags of several source tiles."""
import numpy as np
import pytest
import torch

from test_gpu_chain import _oracle_chain, _t, _to_chain
from unit_amd import chain, ops, rng
from unit_amd._lib import UnitError, check

pytestmark = pytest.mark.gpu

# (oc, (kh, kw), stride, padding, source or None for the layer before)
ODD = [(16, (1, 1), 1, 0, None), (80, (3, 3), 1, 1, None), (48, (5, 5), 2, 2, None), (16, (1, 1), 2, 0, None),
       (16, (1, 1), 1, 0, None), (112, (3, 3), 3, (0, 2, 1, 0), 1), (32, (1, 3), 1, (0, 1, 0, 1), None), (64, (3, 3), 1, 2, 2),
       (144, (1, 1), 1, 0, None), (32, (3, 2), 1, 0, None), (16, (3, 3), 1, 2, None)]
BLOCKS = [(64, (1, 1), 1, 0, None), (64, (3, 3), 1, 1, None), (256, (1, 1), 1, 0, None), (256, (1, 1), 1, 0, -1),
          (64, (1, 1), 1, 0, 2), (64, (3, 3), 1, 1, None), (256, (1, 1), 1, 0, None), (128, (1, 1), 2, 0, 6),
          (128, (3, 3), 1, 1, None), (512, (1, 1), 1, 0, None), (512, (1, 1), 2, 0, 6), (128, (1, 1), 1, 0, 9)]
DEEP = [(256, (3, 3), 1, 1, None), (256, (3, 3), 1, 1, None), (1040, (1, 1), 1, 0, None), (96, (1, 1), 1, 0, None),
        (96, (3, 3), 2, 1, None), (96, (1, 1), 1, 0, None), (96, (1, 1), 1, 0, None), (96, (1, 1), 1, 0, 4),
        (96, (1, 1), 1, 0, 4), (96, (1, 1), 1, 0, 5), (96, (1, 1), 1, 0, None), (96, (1, 1), 1, 0, None)]
# 3 x 3 windows over whole pairs of channel blocks per k-group: strides, uneven and no padding
THREES = [(64, (3, 3), 2, (1, 0, 2, 1), None), (64, (3, 3), 1, 0, None), (128, (3, 3), 1, 1, None), (32, (3, 3), 3, 2, 1),
          (128, (3, 3), 1, (2, 2, 0, 1), None), (64, (3, 3), 1, 1, None), (96, (3, 3), 2, 2, None), (32, (3, 3), 1, 2, None),
          (256, (3, 3), 1, 2, None), (64, (3, 3), 2, 1, None), (32, (3, 3), 1, 1, None), (64, (3, 3), 1, 1, 4)]
WIDE = [(512, (1, 1), 1, 0, None), (1024, (1, 1), 1, 0, None), (1008, (1, 1), 1, 0, 0)] + [(32, (1, 1), 1, 0, None)] * 10
CASES = {
    "odd_blocks_uneven_groups": (ODD, 9, 48, 21, 17),
    "one_image": (ODD, 1, 48, 33, 30),
    "images_smaller_than_a_tile": (ODD, 33, 48, 7, 9),
    "blocks_uneven_groups": (BLOCKS, 17, 64, 14, 13),
    "blocks_one_image": (BLOCKS, 1, 64, 28, 28),
    "wide": (WIDE, 8, 256, 23, 23),
    "threes": (THREES, 12, 32, 27, 30),
    "threes_one_image": (THREES, 1, 32, 30, 27),
    "deep": (DEEP, 3, 128, 9, 8),
    "deep_few_pixels": (DEEP, 64, 128, 3, 3),
}


def _build(oracle, spec, n, c0, h, w, seed=0):
    x = rng.uniform_u8((n, c0 // 16, h, w, 16), 7 + seed)
    layers, outs, chans = [], [], []
    for i, (oc, (kh, kw), stride, pad, source) in enumerate(spec):
        source = i - 1 if source is None else source
        ic = c0 if source < 0 else chans[source]
        wt = rng.uniform_s8((oc, ic, kh, kw), 100 + i)
        b = rng.uniform_s8((oc,), 200 + i).astype(np.int32) * 1000 if i % 2 == 0 else None
        src = x if source < 0 else outs[source]
        acc = oracle.c_conv2d_nchwc(src, oracle.prepack_conv_weight(wt, 16), stride, pad, 1)
        # keeps the activations spread over 0 .. 255; every fourth scale is wide, and its shift long
        scale = 3 if i % 4 else 3 << 20
        shift = max(1, int(np.ceil(np.log2(max(np.percentile(acc, 95), 1.0) * 3 / 200)))) + (0 if i % 4 else 20)
        layers.append((wt, b, scale, shift, stride, pad, source))
        outs.append(_oracle_chain(oracle, [layers[-1][:6] + (-1,)], src)[0])
        chans.append(oc)
    return x, layers, outs


@pytest.mark.parametrize("name", CASES)
def test_chain_kernel_bit_exact(dev, oracle, name):
    spec, n, c0, h, w = CASES[name]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    for _ in range(3):
        for o in c.outputs:
            o.fill_(77)
        c(_t(x, dev))
        for i, (got, ref) in enumerate(zip(c.outputs, want)):
            assert np.array_equal(got.cpu().numpy(), ref), f"layer {i} ({c.variants[i]})"
    assert all(v.startswith("q8chain_") for v in c.variants), c.variants
    assert (want[-1] > 0).mean() > 0.05


def test_chain_kernel_cases_take_every_split(dev):
    kinds = set()
    for spec, n, c0, h, w in CASES.values():
        chans, layers = [], []
        for i, (oc, window, stride, pad, source) in enumerate(spec):
            source = i - 1 if source is None else source
            wt = torch.zeros((oc, c0 if source < 0 else chans[source], *window), dtype=torch.int8, device=dev)
            layers.append(chain.ChainLayer(wt, None, 1, 8, stride, pad, source))
            chans.append(oc)
        c = chain.ConvChain(layers, (n, c0 // 16, h, w, 16))
        c(torch.zeros(c.input_shape, dtype=torch.uint8, device=dev))
        kinds |= {v.split("_")[3] for v in c.variants}
    assert kinds == {"g1", "g2", "g4"}


def test_chain_kernel_replay_and_two_streams(dev, oracle):
    spec, n, c0, h, w = CASES["odd_blocks_uneven_groups"]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    x2 = rng.uniform_u8(x.shape, 99)
    want2 = _oracle_chain(oracle, layers, x2)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    xd = _t(x, dev)
    replay = c.graph(xd)
    for a, ref in ((x, want), (x2, want2), (x, want)):  # the program's own work and synchronisations between the replays
        xd.copy_(_t(a, dev))
        torch.cuda.synchronize()
        replay()
        torch.cuda.synchronize()
        assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(c.outputs, ref))
    # two runs of one chain at once write the same bytes
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(4):
        for s in streams:
            with torch.cuda.stream(s):
                c(xd)
    torch.cuda.synchronize()
    assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(c.outputs, want))


def test_chains_on_two_streams(dev, oracle):
    """Two chains of the same layers on different inputs, run after run on two streams at once: neither sees the other's tickets,
    flags or results."""
    spec, n, c0, h, w = CASES["odd_blocks_uneven_groups"]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    inputs = [x, rng.uniform_u8(x.shape, 99)]
    wants = [want, _oracle_chain(oracle, layers, inputs[1])]
    assert not np.array_equal(wants[0][-1], wants[1][-1])
    chains = [chain.ConvChain(_to_chain(layers, dev), x.shape) for _ in inputs]
    xs = [_t(a, dev) for a in inputs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    kept = [[], []]
    torch.cuda.synchronize()
    for _ in range(6):
        for k in (0, 1):
            with torch.cuda.stream(streams[k]):
                chains[k](xs[k])
                kept[k].append([o.clone() for o in chains[k].outputs])  # every run's, not the last one's only
    torch.cuda.synchronize()
    for k in (0, 1):
        chains[k].check()
        for outs in kept[k]:
            assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(outs, wants[k]))
    assert all(v.startswith("q8chain_") for c in chains for v in c.variants)


def test_chain_with_reused_buffers_runs_layer_by_layer(dev, oracle):
    spec = [(32, (3, 3), 1, 1, None)] * 12
    x, layers, want = _build(oracle, spec, 9, 32, 9, 9)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    c(_t(x, dev))
    assert np.array_equal(c.outputs[-1].cpu().numpy(), want[-1])
    assert all(v.startswith("q8chain_") for v in c.variants)
    for i in range(2, 11):
        c.outputs[i] = c.outputs[i % 2]  # two buffers, written in turn
    c.variants = [None] * 12
    c(_t(x, dev))
    assert np.array_equal(c.outputs[-1].cpu().numpy(), want[-1])
    assert not any(v.startswith("q8chain_") for v in c.variants)


@pytest.mark.parametrize("offset", [0, 16, 64, 112])
def test_workspace_at_any_16_bytes(dev, oracle, offset):
    """The library aligns its own lines inside the workspace and stays within the size that it asked for."""
    spec, n, c0, h, w = CASES["odd_blocks_uneven_groups"]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    xd = _t(x, dev)
    c(xd)
    buf = torch.full((256 + c._ws_bytes + 256,), 0x5A, dtype=torch.uint8, device=dev)
    assert buf.data_ptr() % 128 == 0
    ws = buf[offset:offset + c._ws_bytes]
    for o in c.outputs:
        o.fill_(77)
    check(c._L.unit_conv_chain_u8_ws(c._native, len(c._native), xd.data_ptr(), ws.data_ptr(), c._ws_bytes, ops._stream()))
    torch.cuda.synchronize()
    assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(c.outputs, want))
    assert (buf[:offset] == 0x5A).all() and (buf[offset + c._ws_bytes:] == 0x5A).all()


def test_a_run_that_gives_up_says_so(dev, oracle, monkeypatch):
    """One poll per wave: waits end at once, every kernel still ends by itself, and the run is reported instead of passing for good."""
    spec, n, c0, h, w = CASES["odd_blocks_uneven_groups"]
    x, layers, want = _build(oracle, spec, n, c0, h, w)
    c, other = chain.ConvChain(_to_chain(layers, dev), x.shape), chain.ConvChain(_to_chain(layers, dev), x.shape)
    xd = _t(x, dev)
    replay = c.graph(xd)
    torch.cuda.synchronize()
    c.check()
    monkeypatch.setenv("UNIT_AMD_CHAIN_POLLS", "1")
    c(xd)
    torch.cuda.synchronize()
    other.check()
    with pytest.raises(UnitError, match="gave up"):
        c.check()
    c.check()  # said once
    c(xd)
    torch.cuda.synchronize()
    with pytest.raises(UnitError, match="gave up"):
        c(xd)
    c(xd)
    torch.cuda.synchronize()
    with pytest.raises(UnitError, match="gave up"):
        replay()
    # without a word of the caller's: the workspace's first
    ws = torch.zeros(c._ws_bytes, dtype=torch.uint8, device=dev)
    check(c._L.unit_conv_chain_u8_ws(c._native, len(c._native), xd.data_ptr(), ws.data_ptr(), c._ws_bytes, ops._stream()))
    torch.cuda.synchronize()
    assert ws[:4].view(torch.int32).item() == 1
    monkeypatch.delenv("UNIT_AMD_CHAIN_POLLS")
    ws.zero_()
    check(c._L.unit_conv_chain_u8_ws(c._native, len(c._native), xd.data_ptr(), ws.data_ptr(), c._ws_bytes, ops._stream()))
    torch.cuda.synchronize()
    assert ws[:4].view(torch.int32).item() == 0
    for call in (lambda: c(xd), replay):
        for o in c.outputs:
            o.fill_(77)
        call()
        torch.cuda.synchronize()
        c.check()
        assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(c.outputs, want))


def test_short_chain_takes_no_workspace(dev, oracle):
    """Two layers run launch by launch, with nothing of the kernel's in the way: no workspace, no plan on every run."""
    x, layers, want = _build(oracle, ODD[:2], 2, 48, 21, 17)
    c = chain.ConvChain(_to_chain(layers, dev), x.shape)
    called = []

    class Noted:
        def __getattr__(self, name):
            called.append(name)
            return getattr(lib, name)

    lib, c._L = c._L, Noted()
    c(_t(x, dev))
    assert called == ["unit_conv_chain_u8"]
    assert all(np.array_equal(o.cpu().numpy(), r) for o, r in zip(c.outputs, want))
