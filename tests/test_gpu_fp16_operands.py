"""The fp16 convolution on plain NCHW / OIHW operands: both are re-laid by one kernel before the convolution.  Window
sizes on both sides of the LDS transposition's limit (49 positions), output channels that leave half a 32-channel block
empty, odd images, and operands that start at an odd element."""
import numpy as np
import pytest
import torch

import unit_amd as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W,K,KH,KW,stride,offset", [
    (1, 16, 5, 5, 16, 1, 1, 1, 0),
    (2, 48, 9, 7, 80, 3, 3, 2, 0),
    (3, 16, 1, 5, 32, 1, 2, 1, 1),
    (1, 32, 7, 8, 48, 7, 7, 1, 1),
    (1, 16, 9, 9, 16, 8, 8, 1, 0),
    (2, 32, 31, 33, 64, 5, 5, 2, 3),
])
def test_plain_operands(dev, oracle, N, C, H, W, K, KH, KW, stride, offset):
    g = np.random.RandomState(C + K + KH)
    a = g.randint(-3, 4, (N, C, H, W)).astype(np.float16)
    b = g.randint(-2, 3, (K, C, KH, KW)).astype(np.float16)

    def shifted(x):  # the same values behind `offset` elements: integer data keeps the comparison exact
        t = torch.zeros(x.size + offset, dtype=torch.float16, device=dev)
        t[offset:] = torch.from_numpy(x.reshape(-1)).to(dev)
        return t[offset:].view(x.shape)

    out = U.conv2d_NCHW16c_OHWI16o(shifted(a), shifted(b), stride, stride).cpu().numpy()
    ref = oracle.conv2d_nchw16c_f16(oracle.pack_nchwc(a, 16), oracle.prepack_conv_weight_f16(b), stride, stride)
    assert np.array_equal(out.astype(np.float64), ref), U.last_variant()


def test_weights_at_the_size_limit(dev):
    """2 147 200 000 bytes of weights whose 32-channel form would pass 2^31 - 1."""
    K, C = 10000, 16 * 6710
    g = torch.Generator(device=dev).manual_seed(1)
    a = torch.randint(-1, 2, (1, C, 1, 1), dtype=torch.int8, device=dev, generator=g).half()
    b = torch.randint(-1, 2, (K, C, 1, 1), dtype=torch.int8, device=dev, generator=g).half()
    out = U.conv2d_NCHW16c_OHWI16o(a, b, 1, 1)
    ref = torch.cat([part.reshape(-1, C).float() @ a.reshape(C).float() for part in b.split(2000)])  # exact: sums below 2^24
    assert torch.equal(out.reshape(K), ref), U.last_variant()
