"""GEMMs on the group tiles (gemm_group.hpp): every tile shape with every layout of the second operand, reductions that
end inside a 64-byte stage, row and column edges, N of 4 mod 8 (the transposing read's shifted last chunk), fewer stages
than groups, k-splits by atomics (pinned, and where int8 takes them by itself) and by planes.  Integer data makes the fp16 products exact in any order, so everything is compared bit for bit."""
import numpy as np
import pytest
import torch

import unit_amd as U
from unit_amd import _lib

pytestmark = pytest.mark.gpu

# M, N, K; the tile the shape is there for (fp16 with fp16 output)
F16 = [(1, 8, 8, "x32_y32_k64_w1x1_g4"), (33, 12, 24, "x32_y32"), (37, 36, 200, "x32_y32_k64_w1x1_g8"), (300, 260, 520, "x32_y32"),
       (700, 700, 712, "x32_y64"), (300, 3004, 296, "x64_y64"), (1000, 1516, 1096, "x64_y128"),
       (1500, 1508, 1496, "x128_y128"), (2180, 2052, 2056, "x128_y128"), (3840, 2044, 2056, "x256_y128"), (129, 8192, 40, "")]
# M, N, K; the tile with row-major or prepared weights, and with packed ones (None: N is no multiple of 128)
G4, G8, G4W = "x32_y32_k64_w1x1_g4", "x32_y32_k64_w1x1_g8", "x32_y32_k128_w1x1_g4"
I8 = [(1, 4, 16, G4, None), (33, 36, 80, G4, None), (1, 256, 480, G8, G8), (50, 260, 1040, G4, None), (37, 128, 4112, G4, G4W),
      (64, 4096, 2064, "x32_y32_k64", "x32_y32_k64"), (64, 4096, 3056, "x32_y32_k64", "x32_y32_k64"), (64, 4096, 4096, G4W, G4W),
      (700, 704, 720, "x32_y64", None), (128, 3072, 784, "x32_y64", "x32_y64"),
      (129, 8192, 48, "x64_y64", "x64_y64"), (300, 3072, 304, "x64_y64", "x64_y64"), (1467, 1108, 976, "x64_y128", None),
      (1000, 1536, 1104, "x64_y128", "x64_y128"), (1500, 1536, 1552, "x128_y128", "x128_y128"),
      (2180, 2176, 2064, "x128_y128", "x128_y128"), (1175, 4864, 1632, "x256_y128", "x256_y128"),
      (3840, 2048, 4112, "x256_y128", "x256_y256")]


def _ints(g, lo, hi, shape, dtype, dev):
    return torch.from_numpy(g.randint(lo, hi, shape)).to(dev).to(dtype)


@pytest.mark.parametrize("M,N,K,tile", F16)
def test_fp16_group_tiles(dev, M, N, K, tile):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = a.double() @ b.double()  # exact: |sum| <= 6 K < 2^24
    half = U.gemm_fp16(a, b, "float16")
    name = U.last_variant()
    assert torch.equal(half, ref.half()), name
    assert tile in name, name
    assert torch.equal(U.gemm_fp16(a, b).double(), ref), U.last_variant()
    p = U.prepare_gemm_b(b)
    assert torch.equal(U.gemm_fp16(a, p).double(), ref), U.last_variant()
    assert torch.equal(U.gemm_fp16(a, p, "float16"), ref.half()), U.last_variant()
    assert torch.equal(U.gemm_fp16(a, b, "float16", workspace=True), ref.half()), U.last_variant()
    assert torch.equal(U.gemm_fp16(a, b, workspace=True).double(), ref), U.last_variant()


@pytest.mark.parametrize("M,N,K", [(2900, 2900, 2904), (4096, 4092, 1000), (3000, 3004, 3000)])
def test_fp16_large_ragged_products_stay_staged(dev, M, N, K):
    """Large results whose K no direct tile takes: 256 x 256 tiles, with b by columns and prepared."""
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = a.double() @ b.double()
    for operand in (b, U.prepare_gemm_b(b)):
        assert torch.equal(U.gemm_fp16(a, operand).double(), ref)
        assert "x256_y256" in U.last_variant(), U.last_variant()
        assert torch.equal(U.gemm_fp16(a, operand, "float16"), ref.half())


@pytest.mark.parametrize("M,N,K,packed", [(2048, 8192, 1024, True), (8000, 2048, 2000, True), (8000, 2048, 2000, False)])
def test_int8_large_products_stay_staged(dev, M, N, K, packed):
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    assert torch.equal(U.dense_dotprod(a, U.prepack_dense_weight(w)) if packed else U.dense(a, w), ref)
    assert "x256_y256" in U.last_variant(), U.last_variant()
    assert torch.equal(U.dense(a, U.prepare_dense_weight(w)), ref), U.last_variant()


def test_fp16_infinity_past_a_row(dev):
    """What lies behind a row's end (the next row) must not reach the sums: 0 x inf would be NaN."""
    M, N, K = 40, 44, 72
    a = torch.full((M, K), float("inf"), dtype=torch.float16, device=dev)
    a[::2] = 1
    b = torch.ones((K, N), dtype=torch.float16, device=dev)
    for operand in (b, U.prepare_gemm_b(b)):
        out = U.gemm_fp16(a, operand)
        assert torch.equal(out[::2], torch.full_like(out[::2], K)) and torch.isinf(out[1::2]).all(), U.last_variant()


@pytest.mark.parametrize("M,N,K,tile,packed_tile", I8)
def test_int8_group_tiles(dev, M, N, K, tile, packed_tile):
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    for operand in (w, U.prepare_dense_weight(w)):
        assert torch.equal(U.dense(a, operand), ref), U.last_variant()
        assert tile in U.last_variant() and "dma" not in U.last_variant(), U.last_variant()
    if packed_tile:
        assert torch.equal(U.dense_dotprod(a, U.prepack_dense_weight(w)), ref), U.last_variant()
        assert packed_tile in U.last_variant(), U.last_variant()


@pytest.mark.parametrize("splits", [1, 2, 5])
def test_pinned_k_splits(dev, monkeypatch, splits):
    monkeypatch.setenv("UNIT_AMD_DENSE_SPLITK", str(splits))
    monkeypatch.setenv("UNIT_AMD_GEMM_F16_SPLITK", str(splits))
    M, N, K = 70, 132, 1104
    g = np.random.RandomState(splits)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    for operand in (w, U.prepare_dense_weight(w)):
        assert torch.equal(U.dense(a, operand), ref), U.last_variant()
        assert U.last_variant().endswith(f"_s{splits}")
    w = _ints(g, -128, 128, (256, K), torch.int8, dev)  # packed: K ends inside a stage, the next block's weights follow
    assert torch.equal(U.dense_dotprod(a, U.prepack_dense_weight(w)), (a.double() @ w.double().t()).to(torch.int32))
    assert U.last_variant().endswith(f"_s{splits}")
    h, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = h.double() @ b.double()
    for ws in (None, True):
        assert torch.equal(U.gemm_fp16(h, b, workspace=ws).double(), ref), U.last_variant()
        assert U.last_variant().endswith(f"_s{splits}")


@pytest.mark.parametrize("M,N,K", [(512, 512, 512), (640, 640, 992), (256, 256, 256), (128, 4096, 480)])
def test_fp16_without_planes_runs_whole(dev, M, N, K):
    """A shape for which no planes are planned keeps one workgroup per tile when it comes through the workspace entry
    point: k-splits by atomics, which the plain entry point may choose there, would not give the same bits each time."""
    assert U.gemm_fp16_workspace_bytes(M, N, K) == 0
    g = np.random.RandomState(M + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    assert torch.equal(U.gemm_fp16(a, b, workspace=True).double(), a.double() @ b.double())
    assert U.last_variant().endswith("_s1") or "_s" not in U.last_variant(), U.last_variant()


@pytest.mark.parametrize("M,N,K,layout,splits", [
    (512, 516, 12304, "row_major", 3), (512, 516, 12304, "prepared", 3), (2, 3968, 8800, "packed", 1),
    (2, 3968, 8800, "row_major", 1), (700, 128, 12304, "packed", 9), (1, 128, 16384, "packed", 13),
    (1, 128, 16400, "packed", 13), (130, 384, 16400, "packed", 6),
])
def test_int8_automatic_splits(dev, M, N, K, layout, splits):
    """Where int8 products share a long reduction between workgroups by themselves.  The result starts as garbage: the
    splits add into what their launch has cleared."""
    g = np.random.RandomState(M + N + K)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    out = torch.full((M, N), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    L, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    if layout == "packed":
        wp = U.prepack_dense_weight(w)
        _lib.check(L.unit_dense_dotprod_u8s8s32(a.data_ptr(), wp.data_ptr(), out.data_ptr(), M, N, K, stream))
    elif layout == "prepared":
        p = U.prepare_dense_weight(w)
        _lib.check(L.unit_dense_u8s8s32_prepared(a.data_ptr(), p.w.data_ptr(), p.wsum.data_ptr(), out.data_ptr(), M, N, K, stream))
    else:
        _lib.check(L.unit_dense_u8s8s32(a.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K, stream))
    assert torch.equal(out, (a.double() @ w.double().t()).to(torch.int32)), U.last_variant()
    assert U.last_variant().endswith(f"_s{splits}"), U.last_variant()


@pytest.mark.parametrize("M,N,K", [(733, 1600, 7616), (69, 8964, 5472), (1030, 1024, 6016)])
def test_fp32_results_of_more_than_64_tiles_are_reproducible(dev, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M)
    a, b = torch.randn((M, K), device=dev, generator=g).half(), torch.randn((K, N), device=dev, generator=g).half()
    for operand in (b, U.prepare_gemm_b(b)):
        first = U.gemm_fp16(a, operand)
        assert U.last_variant().endswith("_s1"), U.last_variant()
        assert torch.equal(U.gemm_fp16(a, operand), first)


def test_pins_reach_the_large_staged_tiles(dev, monkeypatch):
    M, N, K = 520, 640, 656
    g = np.random.RandomState(5)
    a, w = _ints(g, 0, 256, (M, K), torch.uint8, dev), _ints(g, -128, 128, (N, K), torch.int8, dev)
    h, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    monkeypatch.setenv("UNIT_AMD_DENSE_SPLITK", "2")
    monkeypatch.setenv("UNIT_AMD_GEMM_F16_SPLITK", "2")
    monkeypatch.setenv("UNIT_AMD_DENSE_VARIANT", "14")
    for call in (lambda: U.dense(a, w), lambda: U.dense_dotprod(a, U.prepack_dense_weight(w))):
        assert torch.equal(call(), ref)
        assert "x256_y256" in U.last_variant() and U.last_variant().endswith("_s2"), U.last_variant()
    for pin, name in (("4", "x256_y256_k128_w4x2"), ("7", ""), ("8", "hybrid_x256_y256_k128_w2x4"), ("9", "hybrid_x256_y128_k128_w2x2")):
        monkeypatch.setenv("UNIT_AMD_GEMM_F16_VARIANT", pin)
        k = K if pin == "4" else 640  # the hybrid tiles take whole stages
        assert torch.equal(U.gemm_fp16(h[:, :k].contiguous(), b[:k].contiguous()).double(), h[:, :k].double() @ b[:k].double())
        assert name in U.last_variant() and (pin != "7" or "hybrid" not in U.last_variant()), U.last_variant()
    monkeypatch.delenv("UNIT_AMD_GEMM_F16_VARIANT")
    m, n, k = 2900, 2900, 2904  # stays on staged tiles
    x, y = _ints(g, -3, 4, (m, k), torch.float16, dev), _ints(g, -2, 3, (k, n), torch.float16, dev)
    assert torch.equal(U.gemm_fp16(x, U.prepare_gemm_b(y)).double(), x.double() @ y.double())
    assert "x256_y256" in U.last_variant() and U.last_variant().endswith("_s2"), U.last_variant()


@pytest.mark.parametrize("M,K", [(300, 600), (1, 640), (129, 8200)])
def test_fp16_four_columns_through_planes(dev, M, K):
    g = np.random.RandomState(M + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, 4), torch.float16, dev)
    ref = a.double() @ b.double()
    assert U.gemm_fp16_workspace_bytes(M, 4, K) > 0
    assert torch.equal(U.gemm_fp16(a, b, workspace=True).double(), ref)
    assert "planes" in U.last_variant(), U.last_variant()
    assert torch.equal(U.gemm_fp16(a, b, "float16", workspace=True), ref.half())


@pytest.mark.parametrize("M,N,K,out,kept", [(4405, 1536, 160, "float16", True), (6000, 704, 640, "float16", True),
                                            (6000, 704, 128, "float16", False), (6000, 704, 672, "float16", False),
                                            (6000, 720, 256, "float16", False), (6000, 704, 256, "float32", False)])
def test_fp16_results_on_128_tiles(dev, M, N, K, out, kept):
    g = np.random.RandomState(M + N + K)
    a, b = _ints(g, -3, 4, (M, K), torch.float16, dev), _ints(g, -2, 3, (K, N), torch.float16, dev)
    ref = (a.double() @ b.double()).to(getattr(torch, out))
    for operand in (b, U.prepare_gemm_b(b)):
        assert torch.equal(U.gemm_fp16(a, operand, out), ref), U.last_variant()
        assert ("dma" in U.last_variant()) == kept, U.last_variant()
