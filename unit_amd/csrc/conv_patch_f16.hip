// 3 x 3 fp16 convolution at stride 1 on prepared weights: pixels pass into the CU once instead of once per window position.
//
// What bounds the direct kernels there (conv_direct.hpp) is delivery into the CU: 256 -> 256 on 16 x 16, batch 32, takes 885
// KB into the CU per 128 channel x 64 pixel tile, a third of it the same pixels once per tap.  Here each of the four waves
// of a workgroup has a quarter of the channel blocks and keeps one block's patch -- the input pixels under the tile's
// windows -- in LDS, the next one's on the way (direct loads, no barrier: a patch belongs to one wave); tiles are 64
// channels x 128 pixels, so that the weights, which stay in registers, are read half as often: 410 KB per workgroup.  One
// wave per SIMD (256 accumulators and a ring of nine weight steps) has nobody to hide its instructions: they stand
// between its MFMAs.  us against the direct kernel's best tile, operands that change from call to call: 32 x 256 x 16 x 16 ->
// 256 12.3 -> 10.8 (with the reads and loads in front of the MFMAs 11.6, with dynamic windows 12.6), 1 x 944 x 47 x 59 -> 608
// 52.8 -> 31.5, 53 x 1120 x 18 x 13 -> 160 57.4 -> 34.3; geometric mean over 40 shapes drawn from those it takes 1.34.
#include "conv_direct.hpp"
#include "conv_plan.hpp"
#include "mma_dma.hpp"

namespace unit {
namespace {

constexpr int kGroups = 4;   // k-groups (waves): each has a quarter of the channel blocks, and its own patches
constexpr int kTX = 2, kTY = 4, kBX = 32 * kTX, kBY = 32 * kTY;
constexpr int kTaps = 9;     // the window is 3 x 3; a ring of nine k-steps of weight fragments is a channel block's
constexpr int kPark = kTX * kTY * 4096;
constexpr int kScratchBytes = 32 * 144 + 128;

struct PatchGeom {
  int N, cc, W, OW, ohw, hw, K, npix;
  int blocks;  // of 64 pixels per patch
  u32 img_bytes, data_bytes;
  FastDiv by_ohw, by_ow, by_hw;
};

// NB: patches of up to 64 NB pixels.  In LDS the two 16-byte halves of a pixel's 16 channels lie in planes of their own: a
// fragment's 32 lanes read 512 consecutive bytes.
template <int NB>
__global__ __launch_bounds__(64 * kGroups, 1) void conv_patch_f16(const char *__restrict__ data, const char *__restrict__ wgt,
                                                                   ConvEpilogue<OpF16>::Params ep, PatchGeom g, GridMap gm) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int kPlane = NB * 1024, kSlot = 2 * kPlane;
  const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int bx, by, split;
  gm.locate(blockIdx.x, bx, by, split);
  const int x0 = bx * kBX, y0 = by * kBY;
  const int c0 = g.cc * wave / kGroups, c1 = g.cc * (wave + 1) / kGroups;  // at least one channel block each
  const int nsteps = g.cc * kTaps;

  // the patch: a run of pixels of the image planes laid end to end, from the first pixel's window row on
  int n0, rem0, oh0, ow0;
  g.by_ohw.divmod(y0, n0, rem0);
  g.by_ow.divmod(rem0, oh0, ow0);
  const int first = oh0 * g.W;
  v4i src;
  {
    const unsigned long long base = (unsigned long long)data;
    src[0] = __builtin_amdgcn_readfirstlane((int)(u32)base);
    src[1] = __builtin_amdgcn_readfirstlane((int)((u32)(base >> 32) & 0xffffu));
    src[2] = __builtin_amdgcn_readfirstlane((int)g.data_bytes);
    src[3] = 0x00020000;
  }
  u32 off[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    int n, pix;
    g.by_hw.divmod(first + i * 64 + lane, n, pix);
    off[i] = n0 + n < g.N ? (u32)(n0 + n) * g.img_bytes + (u32)pix * 32u : 0x80000000u;
  }
  const int mine = wave * 2 * kSlot;  // this wave's two patches, one in use and one on the way
  const u32 slots = (u32)(uintptr_t)(lptr_t)lds + (u32)mine;
  auto fetch_patch = [&](int c, int slot) __attribute__((always_inline)) {
    const u32 to = slots + (u32)(slot * kSlot), from = (u32)(c * g.hw) * 32u;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i < g.blocks) {
        dma_buffer_16(to + i * 1024, off[i], src, from);
        dma_buffer_16(to + kPlane + i * 1024, off[i], src, from + 16);
      }
  };
  fetch_patch(c0, 0);
  __builtin_amdgcn_sched_barrier(0);

  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc((void *)wgt, 0, -1, 0x00020000);
  const u32 lane16 = (u32)lane * 16u;
  u32 wp[kTX];
#pragma unroll
  for (int i = 0; i < kTX; ++i) wp[i] = (u32)(min((x0 >> 5) + i, (g.K - 1) >> 5) * nsteps) * 1024u;
  v4i xf[kTaps][kTX];
  auto fetch_w = [&](auto slot, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kTX; ++i)
      xf[decltype(slot)::value][i] =
          __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + (u32)s * 1024u), 0));
  };
  auto for_taps = [&](auto f) __attribute__((always_inline)) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{});
    f(std::integral_constant<int, 4>{});
    f(std::integral_constant<int, 5>{});
    f(std::integral_constant<int, 6>{});
    f(std::integral_constant<int, 7>{});
    f(std::integral_constant<int, 8>{});
  };
  for_taps([&](auto u) __attribute__((always_inline)) { fetch_w(u, c0 * kTaps + decltype(u)::value); });
  __builtin_amdgcn_sched_barrier(0);
  if (c0 + 1 < c1) fetch_patch(c0 + 1, 1);
  __builtin_amdgcn_sched_barrier(0);

  // LDS offset of this lane's pixels inside a patch (pixels past the last one read the tile's first)
  int pix[kTY];
#pragma unroll
  for (int j = 0; j < kTY; ++j) {
    const int m = y0 + j * 32 + l32;
    int n, rem, oh, ow;
    g.by_ohw.divmod(m < g.npix ? m : y0, n, rem);
    g.by_ow.divmod(rem, oh, ow);
    pix[j] = mine + ((n - n0) * g.hw + oh * g.W + ow - first) * 16 + half * kPlane;
  }

  typename OpF16::acc_t acc[kTX][kTY];
#pragma unroll
  for (int i = 0; i < kTX; ++i)
#pragma unroll
    for (int j = 0; j < kTY; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // Pixel fragments are read one tap ahead, weights nine.  Every turn issues the same loads, also the last one (its
  // weights repeat the last k-step): the waits below count them.
  v4i yf[3][kTY];
  const int row = g.W * 16;
  auto load_y = [&](auto tap, int at, int j) __attribute__((always_inline)) {
    constexpr int T = decltype(tap)::value;
    yf[T % 3][j] = *reinterpret_cast<const v4i *>(lds + (pix[j] + at + (T / 3) * row) + (T % 3) * 16);
  };
  UNIT_WAIT_VMCNT(2 * kTaps);  // the first patch has landed: the ring's weights, at least, are younger
  __builtin_amdgcn_sched_barrier(0);
  int at = 0;  // LDS offset of the patch in use
  u32 wnext = (u32)(min(c0 + 1, c1 - 1) * kTaps) * 1024u;  // the channel block whose weights are fetched
#pragma unroll
  for (int j = 0; j < kTY; ++j) load_y(std::integral_constant<int, 0>{}, at, j);
  for (int c = c0; c < c1; ++c) {
    for_taps([&](auto u) __attribute__((always_inline)) {
      constexpr int T = decltype(u)::value;
      using Next = std::integral_constant<int, (T + 1) % kTaps>;
      const bool more = T + 1 < kTaps || c + 1 < c1;
      if constexpr (T + 1 == kTaps) {
        if (more) {
          // the next block's patch has landed: sixteen or more younger loads (weights) have been issued since; this
          // one's last fragments have been read, and its slot takes the patch after the next
          UNIT_WAIT_VMCNT(2 * (kTaps - 1));
          __builtin_amdgcn_s_waitcnt(0xC07F);
          if (c + 2 < c1) fetch_patch(c + 2, at != 0);
          at = at ? 0 : kSlot;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // a lone wave per SIMD hides an instruction only under an MFMA that is already running: the next tap's reads and the
      // ring's loads stand between the MFMAs
#pragma unroll
      for (int i = 0; i < kTX; ++i)
#pragma unroll
        for (int j = 0; j < kTY; ++j) {
          acc[i][j] = OpF16::mma(xf[T][i], yf[T % 3][j], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0) load_y(Next{}, at, j);
          if (j == kTY - 1)
            xf[T][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + wnext + T * 1024u), 0));
          __builtin_amdgcn_sched_barrier(0);
        }
    });
    wnext = c + 2 < c1 ? wnext + kTaps * 1024u : wnext;
  }

  // the groups' partial tiles meet in LDS; a wave adds up its two blocks in group order
  __syncthreads();
#pragma unroll
  for (int b = 0; b < kTX * kTY; ++b)
    if (b / 2 != wave) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<v4f *>(lds + wave * kPark + ((b * 4 + q) * 64 + lane) * 16) =
            v4f{acc[b / kTY][b % kTY][4 * q], acc[b / kTY][b % kTY][4 * q + 1], acc[b / kTY][b % kTY][4 * q + 2], acc[b / kTY][b % kTY][4 * q + 3]};
    }
  __syncthreads();
  char *scratch = lds + kGroups * kPark + wave * kScratchBytes;
#pragma unroll
  for (int b = 0; b < kTX * kTY; ++b)
    if (b / 2 == wave) {
      v16f total;
#pragma unroll
      for (int r = 0; r < 16; ++r) total[r] = 0;
#pragma unroll
      for (int w = 0; w < kGroups; ++w) {
        if (w == b / 2) {
          total += acc[b / kTY][b % kTY];
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const v4f v = *reinterpret_cast<const v4f *>(lds + w * kPark + ((b * 4 + q) * 64 + lane) * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) total[4 * q + e] += v[e];
          }
        }
      }
      store_block<OpF16>(ep, total, nullptr, 1, x0 + (b / kTY) * 32, y0 + (b % kTY) * 32, lane, scratch);
    }
}

// the longest patch of any tile, in pixels
inline long patch_pixels(const ConvGeom &g) {
  const long rows = (kBY - 2) / g.OW + 2, crossings = g.N > 1 ? (kBY - 2) / (g.OH * g.OW) + 1 : 0;
  return (rows + (g.KH - 1) * (1 + crossings)) * g.W;
}

template <int NB>
int run_patch(const unit_conv_desc *d, const ConvGeom &g, const void *a, const void *w, void *out, hipStream_t s) {
  const char *what = "unit_conv2d_nchw16c_f16f32_prepared";
  constexpr int ring = kGroups * 2 * 2 * NB * 1024, back = kGroups * (kPark + kScratchBytes), lds = ring > back ? ring : back;
  static_assert(lds <= kMaxLds, "patches fit the LDS");
  auto kern = conv_patch_f16<NB>;
  static thread_local bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    allowed = true;
  }
  const int cc = d->C / 16, hw = d->H * d->W;
  const PatchGeom p{d->N, cc, d->W, g.OW, g.OH * g.OW, hw, d->K, g.npix, (int)((patch_pixels(g) + 63) / 64),
                    g.img_bytes, (u32)((size_t)d->N * g.img_bytes), g.by_ohw, g.by_ow, FastDiv::make(hw)};
  const ConvEpilogue<OpF16>::Params ep{out, d->K, g.by_ohw.d, g.npix, g.by_ohw, nullptr, 1, nullptr, 0, 0};
  const int gx = ceil_div(d->K, kBX), gy = ceil_div(g.npix, kBY);
  const GridMap gm = GridMap::make(gx, gy, gx, 1);
  set_variant("f16prep_patch_x%d_y%d_g%d_p%d", kBX, kBY, kGroups, 64 * NB);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(64 * kGroups), lds, s, static_cast<const char *>(a), static_cast<const char *>(w), ep, p, gm);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
}

}  // namespace

// Where it pays: us here / on the direct kernels' tiles, by the kernel that heuristic_plan would take.  A round of 256 tiles costs
// 4.6 us and, per channel block (the wave with the most of them counts), half a microsecond, half as much in the first and in
// the last round, by how full that one is (a workgroup's start and its 128 KB of output meet nobody's arithmetic); weights 0.2 us
// per MB.  Direct tiles: few of 64 x 64 3.2 us + 2.7 per GMAC; one wave per tile 3 us and, per channel block, 0.78 with up to two of
// them per CU, 0.84 with three, 1.22 with four, else 0.32 for each; 128-channel tiles of four groups 4.6 + 0.53, and past 1568
// tiles of 64 x 64 128-channel tiles of one wave are not beaten.  Fitted to 843 random shapes timed both ways: of the 597 it takes
// 5 lose, up to 8 % (geometric mean 0.72); a rule on arithmetic alone lost up to 33 %.  220 tiles of 33 channel blocks 22.1 / 32.3,
// 188 of 21 14.8 / 19.2; the other way 104 of 32 15.0 / 14.3, 212 of 9 12.8 / 10.4, 483 of 18 29.4 / 24.1, 896 of 21, 128-channel
// tiles, 55.2 / 41.6.
bool patch_f16_takes(const unit_conv_desc *d, const ConvGeom &g) {
  const int cc = d->C / 16;
  if (d->sh != 1 || d->sw != 1 || d->KH != 3 || d->KW != 3 || cc < kGroups || patch_pixels(g) > 64 * 8) return false;
  const long tiles = (long)ceil_div(d->K, kBX) * ceil_div(g.npix, kBY), t64 = (long)ceil_div(d->K, 64) * ceil_div(g.npix, 64);
  if (t64 < 392) return 5.9 + 0.37 * cc < 0.97 * (3.2 + 2.7e-9 * g.npix * d->K * cc * 144);
  const bool wide = d->K % 128 == 0;
  if (wide && t64 >= 1568) return false;
  const long rounds = (tiles + 255) / 256, waves = (t64 + 255) / 256;
  const double last = tiles / 256.0 - (rounds - 1);
  const double here = 1 + 4.6 * rounds + (ceil_div(cc, kGroups) * kGroups - 1.5) * (0.5 * rounds - 0.3 + 0.26 * last) +
                      0.2e-6 * d->K * cc * 288;
  const double block = waves <= 2 ? 0.78 : waves == 3 ? 0.84 : waves == 4 ? 1.22 : 0.32 * waves;
  const double direct = wide && waves <= 2 ? 4.6 + 0.53 * cc : 3 + block * cc;
  return here < 0.96 * direct;
}

int conv_f16_patch(const unit_conv_desc *d, const ConvGeom &g, const void *a, const void *w, void *out, hipStream_t s) {
  const long px = patch_pixels(g);
  if (px <= 64 * 4) return run_patch<4>(d, g, a, w, out, s);
  if (px <= 64 * 6) return run_patch<6>(d, g, a, w, out, s);
  return run_patch<8>(d, g, a, w, out, s);
}

}  // namespace unit
