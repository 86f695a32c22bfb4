"""Group tiles with stages of 128 bytes (gemm_group.hpp): every tile with every layout of the second operand, reductions that
end anywhere inside a stage and inside its 64-byte halves, fewer stages than the ring or than groups have, edges of tiles."""
import numpy as np
import pytest
import torch

import unit_amd as U

pytestmark = pytest.mark.gpu


def _ints(g, lo, hi, shape, dtype, dev):
    return torch.from_numpy(g.randint(lo, hi, shape)).to(dev).to(dtype)


# M, N, K (fp16 elements), tile for b by columns (None: 64-byte stages) and for prepared b, fp16 output
F16 = [(70, 260, 808, None, "x32_y32_k128_w1x1_g4_r3"), (129, 1028, 1000, None, "x32_y32_k128_w1x1_g4_r3"),
       (700, 700, 712, "x32_y64_k128_w1x2_g4_r3", "x32_y64_k128_w1x2_g4_r3"),
       (900, 900, 520, "x64_y64_k128_w2x2_g2_r3", "x64_y64_k128_w2x2_g2_r3"),
       (1000, 1516, 1096, None, "x64_y128_k128_w2x2_g2_r3"),  # rows of b end inside lines: from 3 KiB of reduction on
       (1000, 1536, 1096, "x64_y128_k128_w2x2_g2_r3", "x64_y128_k128_w2x2_g2_r3"),
       (800, 1500, 1536, "x64_y128_k128_w2x2_g2_r3", "x64_y128_k128_w2x2_g2_r3"),
       (900, 1660, 1608, "x64_y128_k128_w2x2_g2_r3", "x64_y128_k128_w2x2_g2_r3"),
       (1500, 1508, 1496, "x128_y128_k128_w4x2_g1_r3", "x128_y128_k128_w4x2_g1_r3")]
# M, N, K (bytes), tile with row-major and prepared weights (None: shared between workgroups, 64-byte stages), and with packed ones
I8 = [(65, 512, 1552, None, "x32_y32_k128_w1x1_g4_r3"), (128, 768, 3024, None, "x32_y32_k128_w1x1_g4_r3"),
      (64, 1536, 3088, "x32_y32_k128_w1x1_g4_r3", "x32_y32_k128_w1x1_g4_r3"),
      (330, 1280, 2608, "x32_y64_k128_w1x2_g4_r3", "x32_y64_k128_w1x2_g4_r3"),
      (1000, 1024, 1008, "x64_y64_k128_w2x2_g2_r3", "x64_y64_k128_w2x2_g2_r3"),
      (900, 1664, 1616, "x64_y128_k128_w2x2_g2_r3", "x64_y128_k128_w2x2_g2_r3"),
      (1501, 1536, 1552, "x128_y128_k128_w4x2_g1_r3", "x128_y128_k128_w4x2_g1_r3")]


@pytest.mark.parametrize("M,N,K,by_columns,prepared", F16)
def test_fp16(dev, M, N, K, by_columns, prepared):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = a.double() @ b.double()  # exact: |sum| <= 6 K < 2^24
    for operand, tile in ((b, by_columns), (U.prepare_gemm_b(b), prepared)):
        assert torch.equal(U.gemm_fp16(a, operand, "float16"), ref.half()), U.last_variant()
        assert (tile or "_k64_") in U.last_variant(), U.last_variant()
        assert torch.equal(U.gemm_fp16(a, operand).double(), ref), U.last_variant()


@pytest.mark.parametrize("M,N,K,rows,packed", I8)
def test_int8(dev, M, N, K, rows, packed):
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    for call, tile in ((lambda: U.dense(a, w), rows), (lambda: U.dense(a, U.prepare_dense_weight(w)), rows),
                       (lambda: U.dense_dotprod(a, U.prepack_dense_weight(w)), packed)):
        assert torch.equal(call(), ref), U.last_variant()
        assert (tile or "_k64_") in U.last_variant(), U.last_variant()


def test_fp16_infinity_past_a_row(dev):
    """What lies behind a row's end (the next row) must not reach the sums: 0 x inf would be NaN."""
    M, N, K = 90, 300, 808
    a = torch.full((M, K), float("inf"), dtype=torch.float16, device=dev)
    a[::2] = 1
    b = torch.ones((K, N), dtype=torch.float16, device=dev)
    for operand in (b, U.prepare_gemm_b(b)):
        out = U.gemm_fp16(a, operand, "float16")
        assert torch.equal(out[::2], torch.full_like(out[::2], K)) and torch.isinf(out[1::2]).all(), U.last_variant()
    assert "_k128_" in U.last_variant(), U.last_variant()
