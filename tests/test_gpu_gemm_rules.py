"""Which tiles products take at the lines of the rules: one 256 x 128 tile per CU in 128-byte stages, few tiles, short and long
reductions, ragged edges; exact on small integers."""
import numpy as np
import pytest
import torch

import unit_amd as U
from unit_amd._lib import check, load

pytestmark = pytest.mark.gpu

WIDE = "x256_y128_k128_w4x2_g1_r3"


def _ints(g, lo, hi, shape, dtype, dev):
    return torch.from_numpy(g.randint(lo, hi, shape)).to(dev).to(dtype)


# M, N, K, the tile with b by columns and prepared
@pytest.mark.parametrize("M,N,K,tile", [(2304, 2048, 520, WIDE), (2305, 2044, 392, WIDE), (2304, 2048, 376, "_k64_"), (4090, 2040, 520, WIDE),
                                        (4097, 2048, 520, "x128_y128|x256_y256"), (3300, 1292, 1304, WIDE), (2048, 2432, 1032, WIDE), (2180, 2052, 1016, WIDE),
                                        (562, 320, 1544, "x32_y"), (1365, 64, 1856, "x32_y"), (2562, 5436, 72, "x64_y128|x128_y128"), (130, 72, 512, "")])
def test_fp16(dev, M, N, K, tile):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = a.double() @ b.double()  # exact: |sum| <= 6 K < 2^24
    for operand in (b, U.prepare_gemm_b(b)):
        assert torch.equal(U.gemm_fp16(a, operand).double(), ref), U.last_variant()
        name = U.last_variant()
        assert any(t in name.replace("dmatr", "dma") for t in tile.split("|")), name
        assert torch.equal(U.gemm_fp16(a, operand, "float16"), ref.half()), U.last_variant()


# M, N, K, whether fp32 results share the reduction between workgroups, with b by columns and prepared
@pytest.mark.parametrize("M,N,K,columns,prepared", [(1082, 100, 2456, True, False), (535, 236, 3080, True, False), (121, 1196, 2304, True, False),
                                                    (121, 1196, 2296, False, False), (1461, 60, 2456, False, False)])
def test_fp16_splits(dev, M, N, K, columns, prepared):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = a.double() @ b.double()
    for operand, shared in ((b, columns), (U.prepare_gemm_b(b), prepared)):
        assert torch.equal(U.gemm_fp16(a, operand).double(), ref), U.last_variant()
        assert U.last_variant().endswith("_s1") != shared, U.last_variant()


@pytest.mark.parametrize("M,N,K", [(130, 72, 512), (380, 128, 768), (256, 384, 1024), (640, 640, 768), (512, 768, 768), (520, 768, 1024), (700, 100, 512),
                                   (300, 260, 512), (128, 768, 1528)])
def test_fp16_few_tiles_whole(dev, M, N, K):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    for operand in (b, U.prepare_gemm_b(b)):
        assert torch.equal(U.gemm_fp16(a, operand).double(), a.double() @ b.double()), U.last_variant()
        assert U.last_variant().endswith("_s1") and "dma" not in U.last_variant(), U.last_variant()


# M, N, K, the tile with row-major and prepared weights
@pytest.mark.parametrize("M,N,K,tile", [(2304, 2048, 784, WIDE), (2305, 2044, 1040, WIDE), (2304, 2048, 752, "_k64_"), (4090, 2048, 1040, WIDE),
                                        (2048, 2432, 2064, WIDE), (2180, 2176, 1040, WIDE), (4097, 2048, 784, "x128_y128"), (178, 1336, 1216, "x32_y32"), (636, 420, 1536, "x32_y64"),
                                        (1357, 284, 192, "x32_y32"), (141, 348, 5952, "x32_y32"), (24, 564, 6384, "x32_y32"), (33, 900, 3024, "x32_y32"),
                                        (65, 640, 192, "x32_y32"), (500, 128, 192, ""), (300, 1300, 256, "x32_y"),
                                        (2048, 2048, 320, "x64_y"), (1000, 520, 256, "x64_y64"), (130, 132, 128, "x32_y32"), (300, 260, 128, ""),
                                        (64, 256, 2048, "x32_y32"), (128, 760, 3072, "x32_y"), (130, 200, 3072, "x32_y")])
def test_int8(dev, M, N, K, tile):
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    for operand in (w, U.prepare_dense_weight(w)):
        assert torch.equal(U.dense(a, operand), ref), U.last_variant()
        assert tile in U.last_variant(), U.last_variant()


# both sides of 5 KiB of reduction and of 16 tiles of 128 x 128
@pytest.mark.parametrize("M,N,K,shared", [(7, 896, 5120, True), (7, 896, 5104, False), (30, 2048, 6400, True), (30, 2176, 6400, False)])
def test_packed_splits(dev, M, N, K, shared):
    """The result starts as garbage: the ranges add into what their launch has cleared."""
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    wp, out = U.prepack_dense_weight(w), torch.full((M, N), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    check(load().unit_dense_dotprod_u8s8s32(a.data_ptr(), wp.data_ptr(), out.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, (a.double() @ w.double().t()).to(torch.int32)), U.last_variant()
    assert (int(U.last_variant().rsplit("_s", 1)[1]) > 1) == shared, U.last_variant()


@pytest.mark.parametrize("splits,tile", [(1, WIDE), (2, "x128_y128_k64_"), (3, "x128_y128_k64_")])
def test_pinned_splits_keep_the_estimate_s_tile(dev, monkeypatch, splits, tile):
    """The wide tile is for whole reductions: a pinned count of ranges takes the tile that it was measured with."""
    monkeypatch.setenv("UNIT_AMD_GEMM_F16_SPLITK", str(splits))
    M, N, K = 2304, 2048, 1048
    g = np.random.RandomState(splits)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    for operand in (b, U.prepare_gemm_b(b)):
        assert torch.equal(U.gemm_fp16(a, operand).double(), a.double() @ b.double()), U.last_variant()
        assert tile in U.last_variant() and U.last_variant().endswith(f"_s{splits}"), U.last_variant()


def test_infinity_past_a_row_on_wide_tiles(dev):
    """0 x inf would be NaN: what lies behind a row's end must not reach the sums, in stages of 128 bytes too."""
    M, N, K = 2305, 2044, 392
    a = torch.full((M, K), float("inf"), dtype=torch.float16, device=dev)
    a[::2] = 1
    b = torch.ones((K, N), dtype=torch.float16, device=dev)
    for operand in (b, U.prepare_gemm_b(b)):
        out = U.gemm_fp16(a, operand)
        assert WIDE in U.last_variant(), U.last_variant()
        assert torch.equal(out[::2], torch.full_like(out[::2], K)) and torch.isinf(out[1::2]).all()
