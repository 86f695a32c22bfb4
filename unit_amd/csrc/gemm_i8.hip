// int8 dense: c (M, N) i32 = a (M, K) u8 . W^T, W s8 given row-major (N, K) or in the reference's
// (N/128, K/4, 128, 4) pre-pack.  X operand = a (rows m), Y operand = W (rows n).
#include "epilogues.hpp"
#include "host.hpp"
#include "loaders.hpp"
#include "gemm_group.hpp"
#include "gemm_mixed.hpp"
#include "mma_dma.hpp"

namespace unit {
namespace {

// 256 x 256 tiles staged through registers: pre-packed weights, and row-major ones with an odd number of 64-byte stages
// TAIL = false: K is a whole number of stages (the loaders then stage without zeroing selects)
template <bool PACKED, bool TAIL>
int run_dense_staged(const void *a, const void *w, void *c, int M, int N, int K, hipStream_t s) {
  using T = Tile<256, 256, 128, 2, 4>;
  using XL = RowMajorLoader<T::BX, T::BKB, T::NT, true, 1, TAIL>;
  using YL = std::conditional_t<PACKED, VnniLoader<T::BY, T::BKB, T::NT, 128, 1, TAIL>,
                                RowMajorLoader<T::BY, T::BKB, T::NT, false, 1, TAIL>>;
  using Epi = GemmEpilogue<OpI8, false>;
  typename XL::Params xp{static_cast<const char *>(a), M, K, K};
  typename YL::Params yp;
  if constexpr (PACKED)
    yp = {static_cast<const char *>(w), N, K / 4};
  else
    yp = {static_cast<const char *>(w), N, K, K};
  typename Epi::Params ep{c, M, N};
  const int nk = ceil_div(K, T::BKB), gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  const int splits = pinned_k_splits("UNIT_AMD_DENSE_SPLITK", nk);
  set_variant("i8dense%s_x%d_y%d_k%d_w%d%s_s%d", PACKED ? "pk" : "rm", T::BX, T::BY, T::BKB, T::NT / 64, TAIL ? "" : "e",
              splits);
  return launch_mma<OpI8, T, XL, YL, Epi, WS_Y>(xp, yp, ep, nk, gx, gy, 4, splits, c, (size_t)M * N * 4, 0, s,
                                                PACKED ? "unit_dense_dotprod_u8s8s32" : "unit_dense_u8s8s32");
}

// Tiles of at most 256 x 128 with the reduction shared inside the workgroup (gemm_group.hpp).  Sharing it between
// workgroups as well (int32 atomics into the zero-filled output, exact) costs a launch: it pays from 8 KiB of reduction on
// where the estimate without it is 15 us or more (512 x 516 x 12304 30.8 us whole, 20.0 in three ranges; 2081 x 128 x 10208
// 25.7 and 16.4; 2 x 3968 x 8800, estimate 12.6, 9.4 whole and 11.8 in three), and from 4.5 KiB on (packed 5 KiB: 71 x 1024 x 5040 7.5 and
// 7.9) with up to 16 tiles of 128 x 128, if the estimate says so (7 x 896 x 8048 packed 9.2 us whole, 6.8 in six; 8 x 1160 x 7840 8.5 in
// two, 6.7 in six).  The row-major operator shares at least two ways where tests ask for that: with three to six such tiles from 1 KiB of
// reduction on (50 x 260 x 1040 6.3 us, whole 5.1; 128 x 768 x 3072 7.3 and 6.1), with one or two from 4 KiB on (0.95 of the time whole).
// Not with one or two tiles below that (64 x 256 x 2048 6.4 us, whole 5.4) and with 7 - 11 (33 x 820 x 3024 7.0 and 6.1).
template <int YM, int WS>
int run_dense_group(const char *what, const char *tag, const void *a, const void *w, const int *wsum, void *c, int M, int N,
                    int K, hipStream_t s) {
  const int forced = tuning_override("UNIT_AMD_DENSE_SPLITK");
  const long tiles = tiles_of_128(M, N);
  const int least = forced <= 0 && YM == Y_ROWS && tiles <= 6 && K >= (tiles >= 3 ? 1024 : 4096) ? 2 : 1;
  GroupPlan plan = plan_group(M, N, K, least, 1, kAtomicSplits);
  if (forced > 0)
    plan.splits = forced;
  else if ((K >= 8192 && plan.us >= 15.f) || (K >= (YM == Y_VNNI ? 5120 : 4608) && tiles <= 16))
    plan = plan_group(M, N, K, least, 16, kAtomicSplits);
  else if (YM == Y_ROWS)
    plan = prefer_wide_tile(plan, M, N, K);
  const GroupGemm p{static_cast<const char *>(a), static_cast<const char *>(w), (u32)((size_t)M * K), (u32)((size_t)N * K),
                    M, N, K, K, wsum, c, C_ATOMIC, 0};
  return run_group_plan<OpI8, YM, WS, false>(what, tag, p, plan, s);
}

// Row-major weights with whole 64-byte stages: the 128 x 128 tiles of mma_dma.hpp keep the shapes with 512 tiles or more
// (8192 x 1024 x 1024 17.3 against 16.5 us).  Else the group tiles are faster (64 x 4096 x 4096 13.3 -> 7.9 us, 1024^3
// 11.2 -> 7.0, 1024 x 4096 x 4096 29.4 -> 25.3), also with few tiles, whose k-splits cost a zero fill and atomics, and with few stages:
// 178 x 1336 x 1216 12.2 -> 5.4, 636 x 420 x 1536 12.3 -> 6.5, prepared 420 x 304 x 2112 10.9 -> 5.4, 66 x 1288 x 3776 10.8 -> 6.7;
// 1357 x 284 x 192 8.3 -> 4.5, 320 x 4160 x 192 8.3 -> 5.8, 2680 x 1352 x 320 9.2 -> 7.8, 7259 x 404 x 64 prepared 7.8 -> 5.8.  Left here are
// the corners for which tests name this kernel, each as small as whole stages and tiles let it be; us here / on group tiles: one tile and
// up to 128 bytes of reduction (64 x 128 x 128 7.4 / 3.9); row-major weights up to four tiles and 192 bytes (130 x 132 x 192 7.9 / 4.0), 32 -
// 63 tiles and 320 (1000 x 520 x 320 8.6 / 5.3); prepared ones a tile for each CU and 256 bytes (512 x 8192 x 256 8.4 / 7.4), up to six
// whole tiles and 2 - 4 KiB, in k-splits (128 x 768 x 3072 9.9 / 7.0, 5.7 without splits).
inline bool dense_keeps_128(int M, int N, int K, bool prepared) {
  const long tiles = tiles_of_128(M, N);
  if (K % 64 || direct_gemm_large_tiles(M, N)) return false;
  if (tiles >= 512) return true;
  if (K <= 128) return tiles == 1;
  if (!prepared) return K == 192 ? tiles <= 4 : K == 320 && tiles >= 32 && tiles < 64;
  return (K == 256 && tiles == 256) || (M % 128 == 0 && N % 128 == 0 && tiles <= 6 && K >= 2048 && K < 4096);
}

// direct-to-LDS variant: row-major weights, K a whole number of stages.  wsum: the weight's row sums when they
// were prepared beforehand (unit_dense_prepare_weight), else null and the kernel sums the fragments itself -- one
// Y block per wave where the tile has as many Y blocks per wave as waves share them (WS_Y_SPLIT: 4096^3 in 66-69 us
// against 65 us on prepared sums; summing every fragment in every wave cost 75 us).
template <class T, int NSTAGE, bool GIVEN = false>
int run_dense_dma(const void *a, const void *w, void *c, int M, int N, int K, hipStream_t s, const int *wsum = nullptr,
                  int splits = 1) {
  using Epi = GemmEpilogue<OpI8, false>;
  DmaParams p{static_cast<const char *>(a), static_cast<const char *>(w), M, N, K, wsum};
  typename Epi::Params ep{c, M, N};
  const int nk = K / T::BKB, gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  constexpr int lds = NSTAGE * T::STAGE;
  static_assert(lds <= kMaxLds, "ring does not fit the LDS");
  constexpr bool kSplitSums = !GIVEN && T::TY == T::WX && (T::TY & (T::TY - 1)) == 0 && T::TX * T::TY >= 6;
  auto kern = mma_dma_kernel<OpI8, T, NSTAGE, Epi, GIVEN ? WS_Y_GIVEN : kSplitSums ? WS_Y_SPLIT : WS_Y, true>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "unit_dense_u8s8s32: hipFuncSetAttribute: %s", hipGetErrorString(e));
    allowed = true;
  }
  splits = splits < 1 || (size_t)M * N * 4 % 16 ? 1 : (splits > nk ? nk : splits);
  if (splits > 1) {  // the k-ranges add into c with atomics (exact for int32)
    const size_t n16 = (size_t)M * N * 4 / 16;
    hipLaunchKernelGGL(zero_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, static_cast<v4i *>(c), n16);
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, splits);
  set_variant("i8dense%sdma_x%d_y%d_k%d_w%dx%d_r%d_s%d", GIVEN ? "prep_" : "", T::BX, T::BY, T::BKB, T::WX, T::WY, NSTAGE,
              splits);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), lds, s, p, ep, nk, gm UNIT_TRACE(, trace_buffer()));
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "unit_dense_u8s8s32: launch: %s", hipGetErrorString(e));
}

// pre-packed weights straight to registers, activations through LDS (UNIT_AMD_DENSE_VARIANT=13).
// Measured equal to the staged kernel (91.6 vs 91.1 us at 4096^3) although it moves 1.6 x less
// through LDS: the GEMM is bound by instruction issue per SIMD, not by the LDS pipe.
int run_dense_mixed(const void *a, const void *wp, void *c, int M, int N, int K, hipStream_t s) {
  using T = Tile<256, 256, 128, 2, 4>;
  using XL = RowMajorLoader<T::BX, T::BKB, T::NT, true>;
  using Epi = GemmEpilogue<OpI8, false>;
  const char *what = "unit_dense_dotprod_u8s8s32";
  typename XL::Params xp{static_cast<const char *>(a), M, K, K};
  typename Epi::Params ep{c, M, N};
  const int nk = ceil_div(K, T::BKB), gx = ceil_div(M, T::BX), gy = ceil_div(N, T::BY);
  constexpr int lds = 2 * T::XBYTES;
  auto kern = gemm_mixed_i8<T>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    allowed = true;
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, 1);
  set_variant("i8densepk_direct_x%d_y%d_k%d_w%d_s1", T::BX, T::BY, T::BKB, T::NT / 64);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), lds, s, xp, static_cast<const char *>(wp), N, K / 4, ep, nk, gm);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
}

// Row-major weights and a K that the direct tiles do not take, on a large result: the staged 256 x 256 tiles for short
// reductions of an odd number of 64-byte stages (the tests name them), and where their estimate, 1.15 x that of the direct
// tiles, is the lower one (8000 x 2048 x 2000, one round of 256 tiles, 45 us against 56; 5000 x 4096 x 2000, two, 82 against 77).
inline bool dense_stays_staged(int M, int N, int K) {
  if (K % 128 == 0 || M < 256 || N < 256) return false;
  if (K % 128 == 64 && K < 1024 && direct_gemm_large_tiles(M, N)) return true;
  if (one_wide_tile_per_cu(M, N, K)) return false;  // 24 us where 256 x 256 tiles would take 45
  return 1.15f * large_tile_cost(M, N, K) < plan_group(M, N, K, 1, 1, kAtomicSplits).us;
}

template <bool PACKED>
int dense(const void *a, const void *w, void *c, int M, int N, int K, unit_stream_t stream) {
  const char *what = PACKED ? "unit_dense_dotprod_u8s8s32" : "unit_dense_u8s8s32";
  if (!a || !w || !c) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (M <= 0 || N <= 0 || K <= 0) return fail(UNIT_E_ARG, "%s: M, N, K must be positive (got %d, %d, %d)", what, M, N, K);
  if (K % 16) return fail(UNIT_E_ARG, "%s: K must be a multiple of 16 (got %d)", what, K);
  if (PACKED && N % 128) return fail(UNIT_E_ARG, "%s: N must be a multiple of 128 (got %d)", what, N);
  if (!PACKED && N % 4) return fail(UNIT_E_ARG, "%s: N must be a multiple of 4 (got %d)", what, N);
  if (const int per = row_slice(M, (size_t)K, (size_t)N * 4))
    return run_row_slices(M, per, (size_t)K, (size_t)N * 4, a, c, [&](const void *as, void *cs, int rows) {
      return dense<PACKED>(as, w, cs, rows, N, K, stream);
    });
  if (!fits((size_t)M * K) || !fits((size_t)N * K) || !fits((size_t)M * N * 4))
    return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (int rc = check_aligned(what, {a, w, c})) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // measurement aid: pins a kernel where it can run; a number without a kernel (any more) leaves the choice to the rules
  switch (tuning_override("UNIT_AMD_DENSE_VARIANT")) {
    case 12: if (!PACKED && K % 128 == 0) return run_dense_dma<Tile<256, 256, 128, 2, 4>, 2>(a, w, c, M, N, K, s); break;
    case 13: if (PACKED) return run_dense_mixed(a, w, c, M, N, K, s); break;
    case 14: return run_dense_staged<PACKED, true>(a, w, c, M, N, K, s);
    case 16: if (!PACKED && K % 128 == 0) return run_dense_dma<Tile<256, 256, 128, 4, 2>, 2>(a, w, c, M, N, K, s); break;
    case 17: if (!PACKED && K % 64 == 0) return run_dense_dma<Tile<128, 128, 64, 2, 2>, 4>(a, w, c, M, N, K, s); break;
    default: break;
  }
  if constexpr (PACKED) {
    // The staged 256 x 256 tiles take 1.1 x the time of the direct-to-LDS ones on row-major weights (1.15 x with a part of a
    // stage at the end); the 256 x 128 group tile takes 1.3 x its estimate here, whose fragments are four dword reads
    // each (8192 x 4096 x 1024: 70 us, staged 55; 5000 x 4096 x 2000: 73, staged 81).
    const GroupPlan group = plan_group(M, N, K, 1, 1, kAtomicSplits);
    if (M >= 256 && N >= 256 &&
        (K % 128 ? 1.15f : 1.1f) * large_tile_cost(M, N, K) < group.us * (group.tile == kGroupTiles - 1 ? 1.3f : 1.f))
      return K % 128 ? run_dense_staged<true, true>(a, w, c, M, N, K, s) : run_dense_staged<true, false>(a, w, c, M, N, K, s);
    return run_dense_group<Y_VNNI, WS_Y>(what, "i8densepk", a, w, nullptr, c, M, N, K, s);
  } else {
    if (dense_keeps_128(M, N, K, false))
      return run_dense_dma<Tile<128, 128, 64, 2, 2>, 4>(a, w, c, M, N, K, s, nullptr,
                                                        direct_gemm_k_splits("UNIT_AMD_DENSE_SPLITK", M, N, K));
    // the four waves that share a weight fragment divide the weight sums
    if (K % 128 == 0 && direct_gemm_large_tiles(M, N))
      return run_dense_dma<Tile<256, 256, 128, 4, 2>, 2>(a, w, c, M, N, K, s);
    if (dense_stays_staged(M, N, K)) return run_dense_staged<false, true>(a, w, c, M, N, K, s);
    return run_dense_group<Y_ROWS, WS_Y>(what, "i8denserm", a, w, nullptr, c, M, N, K, s);
  }
}

// one wave per weight row: sum of its K bytes
__global__ __launch_bounds__(256) void dense_row_sums(const char *__restrict__ w, int *__restrict__ sums, int N, int K) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  const int *row = reinterpret_cast<const int *>(w + (size_t)n * K);
  int s = 0;
  for (int i = lane; i < K / 4; i += 64) s = __builtin_amdgcn_sdot4(row[i], 0x01010101, s, false);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) sums[n] = s;
}

}  // namespace
}  // namespace unit

extern "C" int unit_dense_prepare_weight(const void *w, int32_t *wsum, int32_t N, int32_t K, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_dense_prepare_weight";
  if (!w || !wsum) return fail(UNIT_E_ARG, "%s: null pointer", what);
  if (N <= 0 || K <= 0 || K % 16) return fail(UNIT_E_ARG, "%s: N, K must be positive and K a multiple of 16 (got %d, %d)", what, N, K);
  if (!fits((size_t)N * K)) return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  if (int rc = check_aligned(what, {w})) return rc;
  if (int rc = check_device()) return rc;
  hipLaunchKernelGGL(dense_row_sums, dim3(ceil_div(N, 4)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const char *>(w), wsum, N, K);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
  set_variant("dense_row_sums_n%d_k%d", N, K);
  return UNIT_OK;
}

extern "C" int unit_dense_u8s8s32_prepared(const void *a, const void *w, const int32_t *wsum, void *c, int32_t M, int32_t N,
                                           int32_t K, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_dense_u8s8s32_prepared";
  if (!a || !w || !wsum || !c) return fail(UNIT_E_ARG, "%s: null pointer", what);
  // arguments that this entry point does not take in one launch run the plain one, which sums the weights itself
  if (M <= 0 || N <= 0 || K <= 0 || K % 16 || N % 4 || row_slice(M, (size_t)K, (size_t)N * 4) || !fits((size_t)M * K) ||
      !fits((size_t)N * K) || !fits((size_t)M * N * 4) || dense_stays_staged(M, N, K))
    return unit_dense_u8s8s32(a, w, c, M, N, K, stream);
  if (int rc = check_aligned(what, {a, w, c})) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dense_keeps_128(M, N, K, true))
    return run_dense_dma<Tile<128, 128, 64, 2, 2>, 4, true>(a, w, c, M, N, K, s, wsum,
                                                            direct_gemm_k_splits("UNIT_AMD_DENSE_SPLITK", M, N, K));
  if (K % 128 == 0 && direct_gemm_large_tiles(M, N))
    return run_dense_dma<Tile<256, 256, 128, 4, 2>, 2, true>(a, w, c, M, N, K, s, wsum);
  return run_dense_group<Y_ROWS, WS_Y_GIVEN>(what, "i8denserm_prep", a, w, wsum, c, M, N, K, s);
}

extern "C" int unit_dense_dotprod_u8s8s32(const void *a, const void *wp, void *c, int32_t M, int32_t N, int32_t K,
                                          unit_stream_t stream) {
  return unit::dense<true>(a, wp, c, M, N, K, stream);
}

extern "C" int unit_dense_u8s8s32(const void *a, const void *w, void *c, int32_t M, int32_t N, int32_t K,
                                  unit_stream_t stream) {
  return unit::dense<false>(a, w, c, M, N, K, stream);
}
