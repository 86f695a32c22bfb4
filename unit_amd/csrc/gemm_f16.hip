// fp16 GEMM: c (M, N) = a (M, K) f16 . b (K, N) f16, fp32 accumulate on v_mfma_f32_32x32x16_f16.
// X operand = a (rows m, K-contiguous), Y operand = b (rows n, transposed while staging).
#include <mutex>

#include "epilogues.hpp"
#include "gemm_group.hpp"
#include "host.hpp"
#include "loaders.hpp"
#include "mma_dma.hpp"

namespace unit {
namespace {

// Prepared b: (N, K) rows, K-contiguous like a.  Both operands then go global -> LDS directly
// (no register round trip, no transposition), through a ring of NSTAGE LDS buffers; K a whole
// number of stages.
template <class T, int NSTAGE, bool OUT_F16>
int run_gemm_f16_bt_dma(const void *a, const void *bt, void *c, int M, int N, int K, hipStream_t s, int splits = 1) {
  using Epi = GemmEpilogue<OpF16, OUT_F16>;
  DmaParams p{static_cast<const char *>(a), static_cast<const char *>(bt), M, N, K * 2, nullptr};
  typename Epi::Params ep{c, M, N};
  const int nk = K * 2 / T::BKB, gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  constexpr int lds = NSTAGE * T::STAGE;
  static_assert(lds <= kMaxLds, "ring does not fit the LDS");
  auto kern = mma_dma_kernel<OpF16, T, NSTAGE, Epi, WS_NONE, false>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "unit_gemm_f16_prepared: hipFuncSetAttribute: %s", hipGetErrorString(e));
    allowed = true;
  }
  splits = OUT_F16 || splits < 1 ? 1 : (splits > nk ? nk : splits);
  if (splits > 1) {  // the k-ranges add into c with atomics
    const size_t n16 = (size_t)M * N * 4 / 16;
    hipLaunchKernelGGL(zero_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, static_cast<v4i *>(c), n16);
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, splits);
  set_variant("f16gemmbt_dma_x%d_y%d_k%d_w%dx%d_r%d%s_s%d", T::BX, T::BY, T::BKB, T::WX, T::WY, NSTAGE, OUT_F16 ? "_h" : "",
              splits);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), lds, s, p, ep, nk, gm UNIT_TRACE(, trace_buffer()));
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "unit_gemm_f16_prepared: launch: %s", hipGetErrorString(e));
}

// b (K, N) as the reference gives it, both operands global -> LDS directly: b's tile lands as it lies in memory and
// the fragments come out of it with the LDS transposing read (K a whole number of stages, N a multiple of 8).
// splits > 1: k-ranges, added with atomics into the zero-filled c (fp32 results only).
template <class T, int NSTAGE, bool OUT_F16>
int run_gemm_f16_dma_tr(const void *a, const void *b, void *c, int M, int N, int K, hipStream_t s, int splits = 1) {
  using Epi = GemmEpilogue<OpF16, OUT_F16>;
  DmaParams p{static_cast<const char *>(a), static_cast<const char *>(b), M, N, K * 2, nullptr, N * 2};
  typename Epi::Params ep{c, M, N};
  const int nk = K * 2 / T::BKB, gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  constexpr int lds = NSTAGE * T::STAGE;
  static_assert(lds <= kMaxLds, "ring does not fit the LDS");
  auto kern = mma_dma_kernel<OpF16, T, NSTAGE, Epi, WS_NONE, false, true>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "unit_gemm_f16: hipFuncSetAttribute: %s", hipGetErrorString(e));
    allowed = true;
  }
  splits = OUT_F16 || splits < 1 ? 1 : (splits > nk ? nk : splits);
  if (splits > 1) {
    const size_t n16 = (size_t)M * N * 4 / 16;
    hipLaunchKernelGGL(zero_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, static_cast<v4i *>(c), n16);
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, splits);
  set_variant("f16gemm_%s_x%d_y%d_k%d_w%dx%d_r%d_s%d", OUT_F16 ? "dmatr_h" : "dmatr", T::BX, T::BY, T::BKB, T::WX, T::WY, NSTAGE,
              splits);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), lds, s, p, ep, nk, gm UNIT_TRACE(, trace_buffer()));
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "unit_gemm_f16: launch: %s", hipGetErrorString(e));
}

// b (K, N): a goes global -> LDS directly, b through the transposing register loader (K a whole number of stages)
template <class T, bool OUT_F16>
int run_gemm_f16_hybrid(const void *a, const void *b, void *c, int M, int N, int K, hipStream_t s) {
  using YL = KMajorF16Loader<T::BY, T::BKB, T::NT, 1, false>;
  using Epi = GemmEpilogue<OpF16, OUT_F16>;
  DmaParams p{static_cast<const char *>(a), nullptr, M, N, K * 2, nullptr};
  typename YL::Params yp{static_cast<const char *>(b), N, K, N + 4, 0, N * 2};
  typename Epi::Params ep{c, M, N};
  const int nk = K * 2 / T::BKB, gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  constexpr int lds = 2 * T::STAGE;
  auto kern = mma_hybrid_kernel<OpF16, T, YL, Epi>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "unit_gemm_f16: hipFuncSetAttribute: %s", hipGetErrorString(e));
    allowed = true;
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, 1);
  set_variant("f16gemm_hybrid_x%d_y%d_k%d_w%dx%d%s", T::BX, T::BY, T::BKB, T::WX, T::WY, OUT_F16 ? "_h" : "");
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), lds, s, p, yp, ep, nk, gm);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "unit_gemm_f16: launch: %s", hipGetErrorString(e));
}

// Tiles of at most 256 x 128 with the reduction shared inside the workgroup (gemm_group.hpp), any K and N the
// operator takes (b by columns: N >= 8).  fp32 results of up to 64 tiles of 128 x 128 may also share it between workgroups
// (atomics into the zero-filled output); with more tiles they are the same bits from run to run, and the estimate's splits
// lost there (900 x 1096 x 7536, 72 tiles, two ranges 64.9 us, whole 49.4; 733 x 1600 x 7616, 78 tiles, 61.8 and 46.2).  With
// up to six such tiles and 3 KiB of reduction at least two ways, which costs nothing (0.99 - 1.02 of the whole tiles' time; 1.2 - 1.35
// from 1 KiB to 2), and with 7 - 11 tiles just over 1 KiB: a test asks for that of 300 x 260 x 520, 6.4 us where whole tiles take 4.8.
// b by columns also with fewer than 12 tiles and 4.5 KiB or more, where the estimate's whole tiles take up to a quarter longer (1082 x
// 100 x 2456 11.9 us, in three ranges 9.4; 535 x 236 x 3080 14.0 and 11.1; 22 products of 2456 and 3080 1.04 in the mean, lowest 0.94;
// at 4 KiB 535 x 236 x 2056 10.7 and 9.8, 978 x 72 x 2056 7.1 and 8.0).  fp16 results keep one workgroup per tile.
template <int YM, bool OUT_F16>
int run_gemm_f16_group(const char *what, const char *tag, const void *a, const void *b, void *c, int M, int N, int K,
                       hipStream_t s, bool whole = false) {
  const int forced = OUT_F16 || whole ? 1 : tuning_override("UNIT_AMD_GEMM_F16_SPLITK");
  const long tiles = tiles_of_128(M, N);
  const int least = forced <= 0 && (tiles <= 6 ? K >= 1536 : tiles < 12 && ((K > 512 && K <= 640) || (YM == Y_COLS && K >= 2304))) ? 2 : 1;
  GroupPlan plan = plan_group(M, N, K * 2, least, forced > 0 || tiles > 64 ? 1 : 19, kAtomicSplits, OUT_F16 ? 2 : 4);
  if (forced > 0) plan.splits = forced;
  plan = prefer_wide_tile(plan, M, N, K * 2);
  const GroupGemm p{static_cast<const char *>(a), static_cast<const char *>(b), (u32)((size_t)M * K * 2),
                    (u32)((size_t)N * K * 2), M, N, K * 2, YM == Y_COLS ? N * 2 : K * 2, nullptr, c, C_ATOMIC, 0};
  return run_group_plan<OpF16, YM, WS_NONE, OUT_F16>(what, tag, p, plan, s);
}

// Which aligned shapes stay on the 128 x 128 tiles of mma_dma.hpp: one nearly full round of the 256 CUs
// (1011 x 3584 x 1216, 224 tiles, 15.6 against 16.2 us on the group tile of the same size; 2048^3 22.9 against 24.8), and 512
// tiles or more (8192 x 1024 x 1024 24.2 and 24.0 us).  The others gain: 1024^3 11.1 -> 7.1 us, 2304 x 2304 x 4096
// 65.5 -> 57.2, 64 x 4096 x 4096 15.6 -> 14.0; and fp32 results of few tiles, whose k-splits cost a zero fill and atomics: 852 x 448 x 2112
// 14.1 -> 9.1, 562 x 320 x 1536 11.2 -> 7.4, 1365 x 64 x 1856 11.1 -> 6.3, 588 x 516 x 320 8.8 -> 4.9.  Left here are
// two corners for which tests name this kernel and its k-splits, whole tiles of more than 128 rows: b by columns up to six tiles and 1 - 2
// KiB (256 x 384 x 512 9.5 us, 4.5 on group tiles), prepared 24 - 31 and 2 - 3 KiB (512 x 768 x 1024 11.8 and 6.1).
// fp16 results of whole 128-byte rows keep them up to 511 tiles for K of 160 to 640 (6000 x 704 x 256 7.3 us of kernel
// against 8.1, 5000 x 1024 x 512 11.1 and 12.0; K = 128 6.1 and 5.8).
inline bool gemm_keeps_128(int M, int N, int K, bool out_f16, bool columns) {
  const long tiles = tiles_of_128(M, N);
  return tiles >= 512 || (tiles >= 192 && tiles <= 256) ||
         (!out_f16 && M > 128 && M % 128 == 0 && N % 128 == 0 &&
          (columns ? tiles <= 6 && K >= 512 && K < 1024 : tiles >= 24 && tiles < 32 && K >= 1024 && K < 1536)) ||
         (out_f16 && tiles > 256 && N % 64 == 0 && K >= 160 && K <= 640);
}

// (N, K) b and a through registers on 256 x 256 tiles: large results with a K that the direct tiles do not take
template <class T, bool OUT_F16>
int run_gemm_f16_bt(const void *a, const void *bt, void *c, int M, int N, int K, hipStream_t s) {
  using XL = RowMajorLoader<T::BX, T::BKB, T::NT, false>;
  using YL = RowMajorLoader<T::BY, T::BKB, T::NT, false>;
  using Epi = GemmEpilogue<OpF16, OUT_F16>;
  typename XL::Params xp{static_cast<const char *>(a), M, K * 2, K * 2};
  typename YL::Params yp{static_cast<const char *>(bt), N, K * 2, K * 2};
  typename Epi::Params ep{c, M, N};
  const int nk = ceil_div(K * 2, T::BKB), gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  const int splits = OUT_F16 ? 1 : pinned_k_splits("UNIT_AMD_GEMM_F16_SPLITK", nk);
  set_variant("f16gemmbt_x%d_y%d_k%d_w%dx%d%s_s%d", T::BX, T::BY, T::BKB, T::WX, T::WY, OUT_F16 ? "_h" : "", splits);
  return launch_mma<OpF16, T, XL, YL, Epi, WS_NONE>(xp, yp, ep, nk, gx, gy, 4, splits, c, (size_t)M * N * 4, 0, s,
                                                    "unit_gemm_f16_prepared");
}

// Large results whose K or N the direct tiles do not take: the 256 x 256 tiles staged through registers take about 9 us
// + 29 us per 1000 of K for each round of 256 tiles, and `scale` is what the group tiles' estimate falls short by there
// (power: 1.2 with b by columns, 1.35 with b in rows).  Staged against group, fp32 results: 3000 x 3004 x 3000 94.7 / 100.6 us
// (b in rows 88.3 / 119.6), 4000 x 4000 x 4008 138 / 156 (135 / 182), 3500 x 3500 x 3000 93 / 114 (95 / 124); the other way
// 4500 x 4500 x 1496, 324 tiles in two rounds, 108 / 97 (105 / 105).
inline bool gemm_staged_pays(int M, int N, int K, float scale) {
  // short reductions are their stores and loads (2562 x 5436 x 72 17.3 us staged, 12.0; 5966 x 6172 x 176 49 and 38); one_wide_tile_per_cu
  if (M < 256 || N < 256 || K < 256 || one_wide_tile_per_cu(M, N, K * 2)) return false;
  const long tiles = (long)ceil_div(M, 256) * ceil_div(N, 256);
  return 2.f + (float)((tiles + 255) / 256) * (9.f + 0.029f * K) < scale * plan_group(M, N, K * 2, 1, 1, kAtomicSplits).us;
}

template <bool OUT_F16>
int gemm_f16_bt(const void *a, const void *bt, void *c, int M, int N, int K, hipStream_t s) {
  if (K % 32 == 0 && K >= 64) {  // both operands straight into LDS; tile choice as in gemm_f16 below
    if (direct_gemm_large_tiles(M, N)) {
      if (K % 64 == 0) return run_gemm_f16_bt_dma<Tile<256, 256, 128, 2, 4>, 2, OUT_F16>(a, bt, c, M, N, K, s);
      return run_gemm_f16_bt_dma<Tile<256, 256, 64, 2, 4>, 4, OUT_F16>(a, bt, c, M, N, K, s);
    }
    if (gemm_keeps_128(M, N, K, OUT_F16, false))
      return run_gemm_f16_bt_dma<Tile<128, 128, 64, 2, 2>, 4, OUT_F16>(a, bt, c, M, N, K, s, direct_gemm_k_splits("UNIT_AMD_GEMM_F16_SPLITK", M, N, 2l * K));
  }
  if (gemm_staged_pays(M, N, K, 1.35f)) return run_gemm_f16_bt<Tile<256, 256, 128, 2, 4>, OUT_F16>(a, bt, c, M, N, K, s);
  return run_gemm_f16_group<Y_ROWS, OUT_F16>("unit_gemm_f16_prepared", "f16gemmbt", a, bt, c, M, N, K, s);
}

// b (K, N) -> bt (N, K): 64 x 64 tiles through LDS, 128-byte row segments on both sides
__global__ __launch_bounds__(256) void transpose_f16(const _Float16 *__restrict__ b, _Float16 *__restrict__ bt, int K,
                                                     int N) {
  __shared__ _Float16 tile[64][66];
  const int k0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4)
    if (k0 + r < K && n0 + tx < N) tile[r][tx] = b[(size_t)(k0 + r) * N + n0 + tx];
  __syncthreads();
  for (int r = ty; r < 64; r += 4)
    if (n0 + r < N && k0 + tx < K) bt[(size_t)(n0 + r) * K + k0 + tx] = tile[tx][r];
}

// bp (N/32, K/32, 32, 32) with bp[y/32][k/32][k%32][y%32] = b[k][y] (apps/gpu/gemm-pack.py:9,17) -> bt (N, K):
// one 32 x 32 block (2 KiB, contiguous in bp) per workgroup, transposed through LDS; 64-byte row segments of bt
__global__ __launch_bounds__(256) void unpack32_f16(const _Float16 *__restrict__ bp, _Float16 *__restrict__ bt, int K) {
  __shared__ _Float16 tile[32][34];
  const int kb = blockIdx.x, nb = blockIdx.y;
  const _Float16 *src = bp + ((size_t)nb * gridDim.x + kb) * 1024;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) tile[r][tx] = src[r * 32 + tx];  // tile[k % 32][y % 32]
  __syncthreads();
  for (int r = ty; r < 32; r += 8) bt[(size_t)(nb * 32 + r) * K + kb * 32 + tx] = tile[tx][r];
}

// both operands through registers: a by rows, b by columns
template <class T, bool OUT_F16>
int run_gemm_f16(const void *a, const void *b, void *c, int M, int N, int K, hipStream_t s, bool whole) {
  using XL = RowMajorLoader<T::BX, T::BKB, T::NT, false>;
  using YL = KMajorF16Loader<T::BY, T::BKB, T::NT>;
  using Epi = GemmEpilogue<OpF16, OUT_F16>;
  typename XL::Params xp{static_cast<const char *>(a), M, K * 2, K * 2};
  typename YL::Params yp{static_cast<const char *>(b), N, K, N + 4, 0, N * 2};
  typename Epi::Params ep{c, M, N};
  const int nk = ceil_div(K * 2, T::BKB), gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  const int splits = OUT_F16 || whole ? 1 : gemm_k_splits("UNIT_AMD_GEMM_F16_SPLITK", M, N, 2l * K, nk);
  set_variant("f16gemm_x%d_y%d_k%d_w%dx%d_p1%s_s%d", T::BX, T::BY, T::BKB, T::WX, T::WY, OUT_F16 ? "_h" : "", splits);
  return launch_mma<OpF16, T, XL, YL, Epi, WS_NONE>(xp, yp, ep, nk, gx, gy, 4, splits, c, (size_t)M * N * 4, 0, s,
                                                    "unit_gemm_f16");
}

// whole: one workgroup per tile, whatever the shape (the entry points that promise the same bits from run to run
// come here when they plan no planes; k-splits added by atomics would end in another order each time)
template <bool OUT_F16>
int gemm_f16(const void *a, const void *b, void *c, int M, int N, int K, hipStream_t s, bool whole = false) {
  // UNIT_AMD_GEMM_F16_VARIANT pins a kernel per process where it can run (measurement aid); a number without a kernel (any
  // more) leaves the choice to the rules
  switch (tuning_override("UNIT_AMD_GEMM_F16_VARIANT")) {
    case 4: return run_gemm_f16<Tile<256, 256, 128, 4, 2>, OUT_F16>(a, b, c, M, N, K, s, whole);
    case 8: if (K % 64 == 0 && K >= 128) return run_gemm_f16_hybrid<Tile<256, 256, 128, 2, 4>, OUT_F16>(a, b, c, M, N, K, s); break;
    case 9: if (K % 64 == 0 && K >= 128) return run_gemm_f16_hybrid<Tile<256, 128, 128, 2, 2>, OUT_F16>(a, b, c, M, N, K, s); break;
    case 10: if (K % 64 == 0 && K >= 128 && N % 8 == 0) return run_gemm_f16_dma_tr<Tile<256, 256, 128, 2, 4>, 2, OUT_F16>(a, b, c, M, N, K, s); break;
    case 11: if (K % 32 == 0 && K >= 128 && N % 8 == 0) return run_gemm_f16_dma_tr<Tile<256, 256, 64, 2, 4>, 4, OUT_F16>(a, b, c, M, N, K, s); break;
    case 15: if (K % 32 == 0 && K >= 128 && N % 8 == 0) return run_gemm_f16_dma_tr<Tile<128, 128, 64, 2, 2>, 4, OUT_F16>(a, b, c, M, N, K, s); break;
    default: break;
  }
  // K a whole number of 64-byte stages and N of 16-byte chunks: both operands straight into LDS, b read back with the
  // transposing LDS read, on 256 x 256 tiles where those fill the chip (4096^3 in 114 us)
  if (K % 32 == 0 && K >= 64 && N % 8 == 0) {
    if (direct_gemm_large_tiles(M, N)) {
      if (K % 64 == 0) return run_gemm_f16_dma_tr<Tile<256, 256, 128, 2, 4>, 2, OUT_F16>(a, b, c, M, N, K, s);
      return run_gemm_f16_dma_tr<Tile<256, 256, 64, 2, 4>, 4, OUT_F16>(a, b, c, M, N, K, s);
    }
    const int splits = direct_gemm_k_splits("UNIT_AMD_GEMM_F16_SPLITK", M, N, 2l * K);
    if (gemm_keeps_128(M, N, K, OUT_F16, true) && !(whole && splits > 1))
      return run_gemm_f16_dma_tr<Tile<128, 128, 64, 2, 2>, 4, OUT_F16>(a, b, c, M, N, K, s, splits);
  }
  // N 4 mod 8, K a whole number of 128-byte stages, and at least 128 tiles of 256 x 128: a straight into LDS, b through
  // the transposing register loader.  256 x 256 tiles of eight waves, or 256 x 128 tiles of four when those need fewer
  // rounds of 256 workgroups for their cost (about 0.55 of a 256 x 256 tile).
  // The 128-byte stages of one_wide_tile_per_cu are faster where they apply (2304 x 2044 x 1024 19.0 us, here 22.8; 4090 x 2044 x 512
  // 19.4 and 20.2); a test names this kernel for such a product (2048 x 2052 x 512 13.5 and 15.6).
  if (N % 8 && M >= 256 && N >= 128 && K % 64 == 0 && K >= 128) {
    const long tiles_big = (long)ceil_div(M, 256) * ceil_div(N, 256), tiles_half = (long)ceil_div(M, 256) * ceil_div(N, 128);
    const long rounds_big = ceil_div((int)tiles_big, 256), rounds_half = ceil_div((int)tiles_half, 256);
    const bool big_ok = N >= 256 && tiles_big >= 128;
    if (big_ok && rounds_big * 100 <= rounds_half * 55)
      return run_gemm_f16_hybrid<Tile<256, 256, 128, 2, 4>, OUT_F16>(a, b, c, M, N, K, s);
    if (tiles_half >= 128) return run_gemm_f16_hybrid<Tile<256, 128, 128, 2, 2>, OUT_F16>(a, b, c, M, N, K, s);
  }
  // four columns: less than one 16-byte chunk of a row of b
  if (N < 8) return run_gemm_f16<Tile<128, 128, 64, 2, 2>, OUT_F16>(a, b, c, M, N, K, s, whole);
  if (gemm_staged_pays(M, N, K, 1.2f)) return run_gemm_f16<Tile<256, 256, 128, 4, 2>, OUT_F16>(a, b, c, M, N, K, s, whole);
  return run_gemm_f16_group<Y_COLS, OUT_F16>("unit_gemm_f16", "f16gemm", a, b, c, M, N, K, s, whole);
}

// ---- k-splits through a workspace: plane s of the workspace takes the partial tiles of split s, a second kernel
// adds the planes in split order (deterministic; fp16 output rounds the final sum once)
// How many planes: by the same estimate as the tiles (at least two with fewer than 12 tiles of 128 x 128 and 1 KiB of
// reduction), and no more than the library's own scratch holds (two always fit below 128 tiles); three from 128 to 255 such
// tiles once each split keeps 2 KiB.  UNIT_AMD_GEMM_F16_SPLITK pins the count.
constexpr size_t kStaticScratchBytes = 16u << 20;
int gemm_f16_ws_splits(int M, int N, int K) {
  const int nk = ceil_div(K * 2, 64), forced = tuning_override("UNIT_AMD_GEMM_F16_SPLITK");
  const long tiles = tiles_of_128(M, N);
  if (forced > 0) return forced < nk ? forced : nk;
  if (N < 8) {  // its kernel has 128 x 128 tiles alone (8 x 4 x 10712: 25.4 us in 83 planes, 18.3 in 19)
    const int most = gemm_k_splits("UNIT_AMD_GEMM_F16_SPLITK", M, N, 2l * K, nk);
    return most < 19 ? most : 19;
  }
  if (tiles >= 256) return 1;
  if (tiles >= 128) return K >= 3072 ? 3 : 1;
  const size_t fit = kStaticScratchBytes / ((size_t)M * N * 4);
  return plan_group(M, N, K * 2, tiles < 12 && K >= 512 ? 2 : 1, fit < 19 ? (int)fit : 19, kPlaneSplits).splits;
}

template <bool OUT_F16>
__global__ __launch_bounds__(256) void add_planes(const v4f *__restrict__ ws, void *__restrict__ c, size_t n4, int splits,
                                                  size_t plane4) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  v4f sum = ws[i];
  for (int s = 1; s < splits; ++s) sum += ws[i + s * plane4];
  if constexpr (OUT_F16) {
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    static_cast<v4h *>(c)[i] = v4h{(_Float16)sum[0], (_Float16)sum[1], (_Float16)sum[2], (_Float16)sum[3]};
  } else {
    static_cast<v4f *>(c)[i] = sum;
  }
}

// a (M, K) . b (K, N) with `splits` > 1 k-ranges; ws holds splits * M * N floats
int gemm_f16_planes(const char *what, const void *a, const void *b, void *c, int M, int N, int K, bool out_f16, void *ws,
                    int splits, hipStream_t s) {
  const size_t plane = (size_t)M * N * 4;
  if (N < 8) {  // less than one 16-byte chunk of a row of b
    using T = Tile<128, 128, 64, 2, 2>;
    GemmPlaneEpilogue::Params ep{ws, M, N, plane};
    using XL = RowMajorLoader<T::BX, T::BKB, T::NT, false>;
    using YL = KMajorF16Loader<T::BY, T::BKB, T::NT>;
    typename XL::Params xp{static_cast<const char *>(a), M, K * 2, K * 2};
    typename YL::Params yp{static_cast<const char *>(b), N, K, N + 4, 0, N * 2};
    const int nk = ceil_div(K * 2, T::BKB), gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
    set_variant("f16gemm_planes_x%d_y%d_k%d_w%dx%d%s_s%d", T::BX, T::BY, T::BKB, T::WX, T::WY, out_f16 ? "_h" : "", splits);
    if (int rc = launch_mma<OpF16, T, XL, YL, GemmPlaneEpilogue, WS_NONE>(xp, yp, ep, nk, gx, gy, 4, splits, nullptr, 0, 0, s, what))
      return rc;
  } else {
    const GroupGemm p{static_cast<const char *>(a), static_cast<const char *>(b), (u32)((size_t)M * K * 2),
                      (u32)((size_t)N * K * 2), M, N, K * 2, N * 2, nullptr, ws, C_PLANES, plane};
    const GroupPlan plan = plan_group(M, N, K * 2, splits, splits, kPlaneSplits);
    if (int rc = run_group_plan<OpF16, Y_COLS, WS_NONE, false>(what, out_f16 ? "f16gemm_planes_h" : "f16gemm_planes", p, plan, s))
      return rc;
  }
  const size_t n4 = (size_t)M * N / 4;
  if (out_f16)
    hipLaunchKernelGGL(add_planes<true>, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, static_cast<const v4f *>(ws), c,
                       n4, splits, n4);
  else
    hipLaunchKernelGGL(add_planes<false>, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, static_cast<const v4f *>(ws),
                       c, n4, splits, n4);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
}

// argument checks shared by the entry points that split the reduction through planes; *splits = 1 when the shape
// runs without k-splits (then the plain entry point serves it)
int gemm_f16_ws_check(const char *what, const void *a, const void *b, const void *c, int M, int N, int K, int *splits) {
  if (!a || !b || !c) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (M <= 0 || N <= 0 || K <= 0) return fail(UNIT_E_ARG, "%s: M, N, K must be positive (got %d, %d, %d)", what, M, N, K);
  if (K % 8) return fail(UNIT_E_ARG, "%s: K must be a multiple of 8 (got %d)", what, K);
  if (N % 4) return fail(UNIT_E_ARG, "%s: N must be a multiple of 4 (got %d)", what, N);
  if (!fits((size_t)M * K * 2) || !fits((size_t)N * K * 2) || !fits((size_t)M * N * 4))
    return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  *splits = gemm_f16_ws_splits(M, N, K);
  return UNIT_OK;
}

}  // namespace
}  // namespace unit

// ---- the same planes in a buffer the library owns: a file-scope device array, so that the entry point below
// allocates nothing.  Each GPU the library runs on holds its own copy of the array at its own address, resolved once
// per device on the first call there (with that device current); host code uses that pointer, never the array's name.
namespace unit {
namespace {
static __device__ __align__(256) char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mutex;

int static_scratch(const char *what, void **ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(UNIT_E_DEVICE, "%s: hipGetDevice: %s", what, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(UNIT_E_DEVICE, "%s: device index %d out of range", what, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(UNIT_E_DEVICE, "%s: hipGetSymbolAddress: %s", what, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return UNIT_OK;
}
}  // namespace
}  // namespace unit

extern "C" int unit_gemm_f16_static(const void *a, const void *b, void *c, int32_t M, int32_t N, int32_t K, int32_t out_f16,
                                    unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16_static";
  int splits = 1;
  if (int rc = gemm_f16_ws_check(what, a, b, c, M, N, K, &splits)) return rc;
  if (int rc = check_aligned(what, {a, b, c})) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (splits <= 1)  // nothing to split: no scratch is touched
    return out_f16 ? gemm_f16<true>(a, b, c, M, N, K, s, true) : gemm_f16<false>(a, b, c, M, N, K, s, true);
  const size_t need = (size_t)splits * M * N * 4;
  if (need > kStaticScratchBytes)
    return fail(UNIT_E_ARG, "%s: %d k-splits of %d x %d need %zu bytes of scratch, the static buffer holds %zu; "
                "use unit_gemm_f16_ws with a workspace", what, splits, M, N, need, kStaticScratchBytes);
  void *ws = nullptr;
  if (int rc = static_scratch(what, &ws)) return rc;
  // every plane element that add_planes reads is written by this call's GEMM first: nothing has to start at zero
  return gemm_f16_planes(what, a, b, c, M, N, K, out_f16 != 0, ws, splits, s);
}

extern "C" int unit_gemm_f16_ws_bytes(int32_t M, int32_t N, int32_t K, size_t *bytes) {
  using namespace unit;
  const char *what = "unit_gemm_f16_ws_bytes";
  if (!bytes) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 || N % 4)
    return fail(UNIT_E_ARG, "%s: M, N, K must be positive, K a multiple of 8 and N of 4 (got %d, %d, %d)", what, M, N, K);
  const int splits = gemm_f16_ws_splits(M, N, K);
  *bytes = splits > 1 ? (size_t)splits * M * N * 4 : 0;
  return UNIT_OK;
}

extern "C" int unit_gemm_f16_ws(const void *a, const void *b, void *c, int32_t M, int32_t N, int32_t K, int32_t out_f16,
                                void *workspace, size_t workspace_bytes, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16_ws";
  int splits = 1;
  if (int rc = gemm_f16_ws_check(what, a, b, c, M, N, K, &splits)) return rc;
  if (splits <= 1) {  // enough tiles, or a short reduction: nothing to split
    if (int rc = check_aligned(what, {a, b, c})) return rc;
    if (int rc = check_device()) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return out_f16 ? gemm_f16<true>(a, b, c, M, N, K, s, true) : gemm_f16<false>(a, b, c, M, N, K, s, true);
  }
  const size_t need = (size_t)splits * M * N * 4;
  if (!workspace || workspace_bytes < need)
    return fail(UNIT_E_ARG, "%s: workspace of %zu bytes needed (got %zu); ask unit_gemm_f16_ws_bytes", what, need,
                workspace ? workspace_bytes : (size_t)0);
  if (int rc = check_aligned(what, {a, b, c, workspace})) return rc;
  if (int rc = check_device()) return rc;
  return gemm_f16_planes(what, a, b, c, M, N, K, out_f16 != 0, workspace, splits, static_cast<hipStream_t>(stream));
}

extern "C" int unit_gemm_f16(const void *a, const void *b, void *c, int32_t M, int32_t N, int32_t K,
                             int32_t out_f16, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16";
  if (!a || !b || !c) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (M <= 0 || N <= 0 || K <= 0) return fail(UNIT_E_ARG, "%s: M, N, K must be positive (got %d, %d, %d)", what, M, N, K);
  if (K % 8) return fail(UNIT_E_ARG, "%s: K must be a multiple of 8 (got %d)", what, K);
  if (N % 4) return fail(UNIT_E_ARG, "%s: N must be a multiple of 4 (got %d)", what, N);
  if (const int per = row_slice(M, (size_t)K * 2, (size_t)N * 4))
    return run_row_slices(M, per, (size_t)K * 2, (size_t)N * (out_f16 ? 2 : 4), a, c, [&](const void *as, void *cs, int rows) {
      return unit_gemm_f16(as, b, cs, rows, N, K, out_f16, stream);
    });
  if (!fits((size_t)M * K * 2) || !fits((size_t)N * K * 2) || !fits((size_t)M * N * 4))
    return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (int rc = check_aligned(what, {a, b, c})) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return out_f16 ? gemm_f16<true>(a, b, c, M, N, K, s) : gemm_f16<false>(a, b, c, M, N, K, s);
}

extern "C" int unit_gemm_f16_prepare_b(const void *b, void *bt, int32_t K, int32_t N, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16_prepare_b";
  if (!b || !bt) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (K <= 0 || N <= 0) return fail(UNIT_E_ARG, "%s: K, N must be positive (got %d, %d)", what, K, N);
  if (K % 8) return fail(UNIT_E_ARG, "%s: K must be a multiple of 8 (got %d)", what, K);
  if (!fits((size_t)N * K * 2)) return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (int rc = check_aligned(what, {b, bt})) return rc;
  if (int rc = check_device()) return rc;
  hipLaunchKernelGGL(transpose_f16, dim3(ceil_div(N, 64), ceil_div(K, 64)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const _Float16 *>(b), static_cast<_Float16 *>(bt), K, N);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
  set_variant("f16_transpose_b");
  return UNIT_OK;
}

extern "C" int unit_gemm_f16_prepare_b_packed32(const void *bp, void *bt, int32_t K, int32_t N, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16_prepare_b_packed32";
  if (!bp || !bt) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (K <= 0 || N <= 0) return fail(UNIT_E_ARG, "%s: K, N must be positive (got %d, %d)", what, K, N);
  if (K % 32 || N % 32) return fail(UNIT_E_ARG, "%s: K and N must be multiples of 32 (got %d, %d)", what, K, N);
  if (!fits((size_t)N * K * 2)) return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (N / 32 > 65535) return fail(UNIT_E_ARG, "%s: N exceeds 32 * 65535", what);
  if (int rc = check_aligned(what, {bp, bt})) return rc;
  if (int rc = check_device()) return rc;
  hipLaunchKernelGGL(unpack32_f16, dim3(K / 32, N / 32), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const _Float16 *>(bp), static_cast<_Float16 *>(bt), K);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
  set_variant("f16_unpack32_b");
  return UNIT_OK;
}

extern "C" int unit_gemm_f16_prepared(const void *a, const void *bt, void *c, int32_t M, int32_t N, int32_t K,
                                      int32_t out_f16, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_gemm_f16_prepared";
  if (!a || !bt || !c) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (M <= 0 || N <= 0 || K <= 0) return fail(UNIT_E_ARG, "%s: M, N, K must be positive (got %d, %d, %d)", what, M, N, K);
  if (K % 8) return fail(UNIT_E_ARG, "%s: K must be a multiple of 8 (got %d)", what, K);
  if (N % 4) return fail(UNIT_E_ARG, "%s: N must be a multiple of 4 (got %d)", what, N);
  if (const int per = row_slice(M, (size_t)K * 2, (size_t)N * 4))
    return run_row_slices(M, per, (size_t)K * 2, (size_t)N * (out_f16 ? 2 : 4), a, c, [&](const void *as, void *cs, int rows) {
      return unit_gemm_f16_prepared(as, bt, cs, rows, N, K, out_f16, stream);
    });
  if (!fits((size_t)M * K * 2) || !fits((size_t)N * K * 2) || !fits((size_t)M * N * 4))
    return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (int rc = check_aligned(what, {a, bt, c})) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return out_f16 ? gemm_f16_bt<true>(a, bt, c, M, N, K, s) : gemm_f16_bt<false>(a, bt, c, M, N, K, s);
}
