"""Layout kernels on both sides of their dispatch lines: planes smaller than a four-byte word of pixels, planes of odd
size (words at any byte address, the last one moved back), and tensors on either side of the line from which packing
takes sixteen pixels per thread."""
import numpy as np
import pytest
import torch

import unit_amd as U
from unit_amd import _lib, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,cb,dtype", [
    ((2, 3, 1, 3), 4, np.uint8), ((2, 5, 1, 5), 4, np.uint8), ((3, 3, 61, 43), 4, np.int8),
    ((2, 33, 1, 2), 16, np.uint8), ((2, 33, 2, 2), 16, np.uint8), ((7, 320, 9, 11), 16, np.int8),
    ((5625, 250, 3, 5), 16, np.uint8),    # 90000 planes of 15 pixels: partial groups of the sixteen-pixel kernel
    ((22499, 16, 4, 4), 16, np.uint8),    # 89996 four-pixel groups
    ((22500, 16, 4, 4), 16, np.uint8),    # 90000
    ((70001, 16, 1, 1), 16, np.uint8), ((70001, 17, 1, 3), 16, np.int8), ((70001, 16, 1, 1), 16, np.int32),
    ((70001, 16, 1, 2), 16, np.float16), ((70001, 3, 1, 4), 4, np.uint8), ((11, 7, 3, 5), 6, np.float16),
    ((110, 24, 1, 220), 16, np.float16), ((400, 32, 7, 7), 16, np.int32),   # both sides of 600000 elements: 774400 and
    ((300, 32, 7, 7), 16, np.float16), ((38000, 16, 1, 1), 16, np.int32),   # 627200, 470400 and 608000
    ((1700, 32, 7, 7), 16, np.int32), ((1500, 64, 1, 26), 16, np.int32),    # 2.67 million by plane, 2.50 million flat
    ((2, 20, 3, 7), 16, np.float16), ((2, 20, 1, 1), 16, np.float16), ((1, 20, 3, 3), 16, np.int32),
])
def test_pack_and_back(dev, oracle, shape, cb, dtype):
    x = rng.random_bytes(int(np.prod(shape)) * np.dtype(dtype).itemsize, 7).view(dtype).reshape(shape)
    if dtype == np.float16:
        x = np.nan_to_num(x, nan=1.0)
    p = U.pack_nchwc(torch.from_numpy(x).to(dev), cb)
    assert np.array_equal(p.cpu().numpy().view(np.uint8), oracle.pack_nchwc(x, cb).view(np.uint8))
    assert np.array_equal(U.unpack_nchwc(p, shape[1]).cpu().numpy().view(np.uint8), x.view(np.uint8))


@pytest.mark.parametrize("shape,cb,dtype", [((2, 20, 3, 5), 16, np.float16), ((3, 3, 5, 7), 4, np.uint8), ((2, 18, 5, 5), 16, np.int8),
                                            ((3, 18, 1, 3), 16, np.int8)])
def test_blocked_tensor_at_an_odd_element(dev, oracle, shape, cb, dtype):
    """The blocked side of the word kernels is read and written in aligned words: other addresses go element by element."""
    x = rng.random_bytes(int(np.prod(shape)) * np.dtype(dtype).itemsize, 8).view(dtype).reshape(shape)
    want = oracle.pack_nchwc(x, cb)
    room = torch.zeros(want.size + 1, dtype=torch.from_numpy(x).dtype, device=dev)
    room[1:] = torch.from_numpy(want.reshape(-1)).to(dev)
    back = U.unpack_nchwc(room[1:].view(want.shape), shape[1])
    assert np.array_equal(back.cpu().numpy().view(np.uint8), x.view(np.uint8))
    room.zero_()
    xd = torch.from_numpy(x).to(dev)
    code = _lib.load().unit_pack_nchwc(xd.data_ptr(), room[1:].data_ptr(), *shape, cb, x.itemsize,
                                       torch.cuda.current_stream().cuda_stream)
    assert code == 0 and np.array_equal(room[1:].cpu().numpy().view(np.uint8), want.reshape(-1).view(np.uint8)) and room[0] == 0
