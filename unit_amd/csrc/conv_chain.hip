// A chain of requantising convolutions (unit_conv_chain_u8) inside one persistent kernel.
//
// What bounds a chain of launches: a layer of a residual network at batch 32 is 6.5 - 14 us of which the launch gap, the
// argument fetch, the decode, the first loads from cold L2s and the last write-back are 4 - 5 us, fifty-two times over
// (ResNet-50 behind its stem: 491 us; at batch 1, where nothing else is left, 219 us).  Here
//   * the images are dealt to the XCDs in groups (batch / 8 each), and an XCD takes its group through all layers: what a
//     layer writes, the next one reads from the same L2, with no write-back and no cold cache in between;
//   * a layer's tile waits for the tiles of its source layer that it reads, not for the layer: a flag per tile, set when
//     the tile's results have reached the L2 (a message from one workgroup to another through the L2 takes 0.2 us; a
//     kernel boundary 1.2 - 1.5 us and the caches);
//   * the weights of a tile, which depend on no other tile, are under way while it waits.
// Measured against the launches, us a pass among others, its setup included: ResNet-50 batch 32 on inputs and buffers that
// change 350 / 491; on two inputs in turn 151 / 219 at batch 1, 171 / 282 at 8, 237 / 331 at 16; ResNet-18 62 / 88 at 1, 79 / 126 at
// 16, 107 / 156 at 32.  At batch 32 the matrix pipes are busy 16 % of the time and a CU takes in 20 bytes of operands per clock:
// what is left is the latency of fifty-two layers, 3 us each at batch 1 (0.6 - 0.8 decode, 0.3 until the flag is seen, 0.8 - 1.4
// loads and reduction, 0.5 k-group sum, requantisation and stores, 0.2 their acknowledgement, 0.2 flag).
//
// Tiles are handed out by a ticket counter per XCD, in the order of the layers.  A workgroup that holds a ticket runs, and
// everything its tile waits for has an earlier ticket, so the earliest unfinished tile never waits: the kernel ends
// whatever part of the grid the device keeps resident.  Groups are claimed, not assigned: an XCD that runs out of
// tickets takes the next group, so the work is done also where some XCD has no workgroup at all.
//
// A wave reads the results of other CUs of its XCD with agent-scope (sc1) loads, which pass the CU's vector cache by and
// hit in the L2 (188 clocks against 108 for a hit in the vector cache); plain loads could return a line that the CU
// fetched before its neighbour wrote it, and dropping the vector cache with buffer_inv sc1 holds up the CU's other loads (1190 us
// for the ResNet-50 above).  Stores and flags are plain: they stay in the L2 (an sc1 store goes to memory, and a load
// after it with it).
//
// The tile: four waves of 64 channels x 64 pixels, 64 x 32 or 32 x 32 each, operands straight into registers as in conv_direct.hpp,
// either side by side (over channels first, then pixels) or in two or four k-groups that share a tile.  With 64 x 64 alone the
// layers behind the second stage of a ResNet keep 8 - 26 of an XCD's 64 workgroups busy at an image per XCD, for up to 5 us each.
#include "conv_direct.hpp"
#include "conv_prepare.hpp"
#include "host.hpp"

#include <algorithm>

namespace unit {

int conv_sizes(const unit_conv_desc *d, int tapb, ConvGeom *g, const char *what);  // abi.hip

namespace {

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kPerCu = 2;                 // workgroups per CU: 256 VGPRs (three of 168 with three k-steps in flight: 392 us at batch 32, 234 at 8)
// A wave's tile is TX x TY blocks of 32 channels x 32 pixels: 2 x 2, 2 x 1 or 1 x 1.  k-steps of fragments in flight per wave: few
// blocks are few MFMAs per step, so more steps to cover a load's latency (nine for one block, a period of chain_reduce_3x3; nine for
// two blocks spilled).  A wave whose share of a 1 x 1 layer is short loads no more than kShort steps.
template <int TX, int TY> constexpr int kRing = TX * TY == 4 ? 5 : TX == 1 ? 9 : 6;
template <int TX, int TY> constexpr int kMaxRing = TX * TY == 4 ? 5 : 9;  // with chain_reduce_patch's, which needs no pixels in registers
template <int TX, int TY> constexpr int kShort = TX * TY == 4 ? 2 : 4;
constexpr int kMaxXcd = 16, kMaxChain = 256;
constexpr int kAgent = 16;        // sc1
// Polls a wave may spend in all before it stops waiting (seconds; a whole chain takes some thousand): every wave ends, also
// after a fault in another one.  A wave that stops waiting says so in the status word: the run's results are then
// not valid.  UNIT_AMD_CHAIN_POLLS sets another number (a test takes one).
constexpr int kPolls = 1 << 24;

// q = n / d for n * d < 2^31 (a double's quotient is exact enough: 2^31 / d is at least 1 / d below the next whole number)
inline u32 small_div(int d) { return (u32)(2147483648.0 / d) + (d != 1); }
__device__ __forceinline__ int quot(int n, u32 mul) { return (int)__umulhi((u32)n << 1, mul); }

// A layer as the kernel reads it.  Sizes are those of a group of images.
struct alignas(128) ChainStep {
  const char *data, *w;
  char *out;
  const int *bias;
  int first, next;  // its tickets in a group's program; a tile's flag has the ticket's number
  int scale, K, nsteps, ntaps, ohw, img_bytes;
  u32 by_ohw, by_ow, by_win, by_kw, by_nct;  // small_div
  int nct;                                   // channel tiles; a pixel tile's are neighbours
  int src_first, src_nct;                    // the source layer's first ticket and channel tiles
  u32 row_ones;                              // ConvGeom
  unsigned short H, W, OW;
  unsigned char pt, pl, KH, KW, sh, sw;
  unsigned char shift, win, mode;  // KH * KW; MODE of the reduction
  unsigned char flat;              // 1 x 1 at stride 1: output pixels are input pixels
  unsigned char reads, src_shift;  // the source is a layer of the chain, its pixel tiles are 1 << src_shift
  unsigned char kg_log, wx_log, wy_log, tile;  // tile: log2 of a wave's channels and, in the upper half, of its pixels
};
static_assert(sizeof(ChainStep) == 128, "ChainStep");
using StepPtr = const __attribute__((address_space(4))) ChainStep *;
// a layer's 128 bytes as two scalar loads of a cache line each
__device__ __forceinline__ ChainStep load_step(StepPtr p) {
  const auto *q = (const __attribute__((address_space(4))) v16i *)p;
  struct alignas(128) Raw {
    v16i a, b;
  } r{q[0], q[1]};
  return __builtin_bit_cast(ChainStep, r);
}

// The workspace: control words (zeroed by chain_setup), then the layers.  Words: groups claimed; a line per XCD with its
// ticket counter; per XCD the groups it has claimed (+ 1), in its order; per group the tiles' flags.  No line of it is
// written by two XCDs but the first, so it begins on a line wherever the caller's memory does (kWsAlign).
constexpr int kWsAlign = 128, kWsHead = 16;  // kWsHead: the status word of callers without one of their own
constexpr int kCtlGroups = 0, kCtlTickets = 32, kCtlSlots = kCtlTickets + 32 * kMaxXcd;

struct ChainArgs {
  const ChainStep *steps;  // the first layer's; the entry in front of it holds the status word's address (give_up)
  int *ctl;
  int polls, images, per, groups;
  int slot_pitch, flags0, flag_pitch;
  FastDiv by_tickets;
};

// The layers travel as kernel arguments (at most 4 KiB of them), so that a captured chain keeps the ones it was captured
// with, and nothing is copied from host memory.
constexpr int kSetupSteps = 31;
struct ChainSetup {
  ChainStep s[kSetupSteps];
};

__global__ __launch_bounds__(256) void chain_setup(const ChainSetup a, ChainStep *steps, int count, v4i *clear, int nclear) {
  if (blockIdx.x == 0 && threadIdx.x < count * 8)
    reinterpret_cast<v4i *>(steps)[threadIdx.x] = reinterpret_cast<const v4i *>(a.s)[threadIdx.x];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < nclear; i += gridDim.x * 256) clear[i] = v4i{0, 0, 0, 0};
}

struct alignas(16) ChainLds {
  v4i part[kWaves][16][64];  // [wave][quad of its blocks][lane]: partial sums for their owners; before them, a wave's pixels
  int addend[kWaves][64];
  int ticket[2], group;
};

// The caller's status word, in device or pinned host memory: 1 once a wave has given up waiting, else as it was.  Its address
// travels as one more step: as a kernel argument it cost registers, and a run 2 us.
__device__ __forceinline__ void give_up(const ChainArgs &a) {
  int *const status = reinterpret_cast<int *>(a.steps[-1].out);
  __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ int load_l2(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// a step's pointers come out of scalar registers: told to be global memory, or every load through them is a flat one
template <class T>
using Global = const __attribute__((address_space(1))) T *;

// MODE 0: one tap per channel block, an even number of them, no padding; 1: any window without padding; 2: any window
struct TapWalk {
  int ntaps, KW, win, row_skip, ch_skip, hw16, w16;
  u32 by_win, by_kw;
};

template <class F, int... U>
__device__ __forceinline__ void for_each_slot(F f, std::integer_sequence<int, U...>) {
  (f(std::integral_constant<int, U>{}), ...);
}

// TX x TY blocks, D k-steps in flight; ONCE: the wave's share is at most D steps
template <int MODE, int TX, int TY, int D, bool ONCE>
__device__ __forceinline__ void chain_reduce(v16i (&acc)[TX][TY], __amdgpu_buffer_rsrc_t wbuf, const u32 (&wp)[TX], __amdgpu_buffer_rsrc_t data, const u32 lane16,
                                             int (&pixoff)[TY], const u32 (&inside)[TY], v4i (&xf)[kMaxRing<TX, TY>][TX], int half, int s0, int s1,
                                             int slast, const TapWalk &tw) {
  v4i yf[D][TY];
  auto for_slots = [&](auto f) __attribute__((always_inline)) { for_each_slot(f, std::make_integer_sequence<int, D>{}); };
  // The state of the running tap; it advances by a k-step per fetch and stops at the wave's last one.  Uniform and
  // without branches, so that the loads keep one order on all paths.
  int sf = s0;
  int kw = 0, pos = 0, off = 0;
  if constexpr (MODE != 0) {
    const int t = 2 * s0, ci = quot(t, tw.by_win);
    pos = t - ci * tw.win;
    const int kh = quot(pos, tw.by_kw);
    kw = pos - kh * tw.KW;
    off = ci * tw.hw16 + kh * tw.w16 + kw * 16;
  } else {
    off = 2 * s0 * tw.hw16;
#pragma unroll
    for (int j = 0; j < TY; ++j) pixoff[j] += half ? tw.hw16 : 0;
  }
  auto fetch_d = [&](auto slot) __attribute__((always_inline)) {
    constexpr int U = decltype(slot)::value;
    if constexpr (MODE == 0) {
#pragma unroll
      for (int j = 0; j < TY; ++j)
        yf[U][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(data, pixoff[j], off, kAgent));
      const bool more = sf < slast;
      sf += more;
      off += more ? 2 * tw.hw16 : 0;
    } else {
      int k2 = kw, p2 = pos, o2 = off;
      auto step = [&]() __attribute__((always_inline)) {
        ++k2, ++p2, o2 += 16;
        const bool cr = k2 == tw.KW;
        k2 = cr ? 0 : k2;
        o2 += cr ? tw.row_skip : 0;
        const bool cc = p2 == tw.win;
        p2 = cc ? 0 : p2;
        o2 += cc ? tw.ch_skip : 0;
      };
      step();
      const bool odd = 2 * sf + 1 < tw.ntaps;
      const int o = half ? (odd ? o2 : off) : off, ps = half ? (odd ? p2 : 31) : pos;
#pragma unroll
      for (int j = 0; j < TY; ++j) {
        u32 v = (u32)(pixoff[j] + o);
        if constexpr (MODE == 2) v |= ~(u32)__builtin_amdgcn_sbfe((int)inside[j], (u32)ps, 1u);
        yf[U][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(data, (int)v, 0, kAgent));
      }
      step();
      const bool more = sf < slast;
      sf += more;
      kw = more ? k2 : kw, pos = more ? p2 : pos, off = more ? o2 : off;
    }
  };
  auto consume = [&](auto slot) __attribute__((always_inline)) {
    constexpr int U = decltype(slot)::value;
    v4i y[TY];
#pragma unroll
    for (int j = 0; j < TY; ++j)
#pragma unroll
      for (int d = 0; d < 4; ++d) y[j][d] = yf[U][j][d] ^ (int)0x80808080;
#pragma unroll
    for (int i = 0; i < TX; ++i)
#pragma unroll
      for (int j = 0; j < TY; ++j) acc[i][j] = OpI8::mma(xf[U][i], y[j], acc[i][j]);
  };
  for_slots([&](auto u) __attribute__((always_inline)) { fetch_d(u); });
  __builtin_amdgcn_sched_barrier(0);
  u32 sw = (u32)min(s0 + D, slast) * 1024u;
  const u32 swlast = (u32)slast * 1024u;
  auto round = [&]() __attribute__((always_inline)) {
    for_slots([&](auto u) __attribute__((always_inline)) {
      consume(u);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int U = decltype(u)::value;
#pragma unroll
      for (int i = 0; i < TX; ++i) xf[U][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + sw), 0));
      sw = min(sw + 1024u, swlast);
      fetch_d(u);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  int s = s0;
  if constexpr (!ONCE) {
    if (s + D < s1) {
      round();
      for (s += D; s + D < s1; s += D) round();
    }
  }
  for_slots([&](auto u) __attribute__((always_inline)) {
    if (s + decltype(u)::value < s1) consume(u);
    __builtin_amdgcn_sched_barrier(0);
  });
}

// MODE 3: 3 x 3 windows, padded or not, and a share of whole periods of nine k-steps (two channel blocks).  The taps of
// a period are known here: an offset and a mask bit per lane and step, set up once, instead of a walk per step; and the
// loads of the ring stand between the MFMAs, where a wave's other instructions cost nothing.  us with the walk of MODE 2 /
// here: ResNet-50 batch 1 213 / 201, 16 252 / 241, 32 389 / 380; ResNet-18 106 / 98 at 16, 133 / 119 at 32.  Loads between the
// MFMAs of the other modes give under 1 % at 1 x 1 windows and take 3 % at ResNet-18, batch 32.  A ring of six in a period of 18 spilled.
template <int TX, int TY> constexpr int kRing3 = TX * TY != 1 ? 3 : 9;
template <int TX, int TY>
__device__ __forceinline__ void chain_reduce_3x3(v16i (&acc)[TX][TY], __amdgpu_buffer_rsrc_t wbuf, const u32 (&wp)[TX],
                                                 __amdgpu_buffer_rsrc_t data, const u32 lane16, const int (&pixoff)[TY],
                                                 const u32 (&inside)[TY], v4i (&xf)[kMaxRing<TX, TY>][TX], int half, int s0, int s1,
                                                 int hw16, int w16) {
  constexpr int D = kRing3<TX, TY>, P = 9;
  static_assert(P % D == 0 && D <= kRing<TX, TY>, "the ring's slots repeat with the period");
  // offset of tap 2 s + half of a period; all ones, out of range, outside the image
  u32 at[9][TY];
#pragma unroll
  for (int s = 0; s < 9; ++s) {
    const int e = 2 * s, o = 2 * s + 1;
    const int oe = (e / 9) * hw16 + (e % 9 / 3) * w16 + (e % 9 % 3) * 16, oo = (o / 9) * hw16 + (o % 9 / 3) * w16 + (o % 9 % 3) * 16;
#pragma unroll
    for (int j = 0; j < TY; ++j)
      at[s][j] = (u32)(pixoff[j] + (half ? oo : oe)) | ~(u32)__builtin_amdgcn_sbfe((int)inside[j], (u32)(half ? o % 9 : e % 9), 1u);
  }
  v4i yf[D][TY];
  int soff = 2 * (s0 / 9) * hw16;
  u32 sw = (u32)s0 * 1024u;
  auto load_d = [&](int s, int j) __attribute__((always_inline)) {
    yf[s % D][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(data, (int)at[s % 9][j], soff + s / 9 * (2 * hw16), kAgent));
  };
#pragma unroll
  for (int s = 0; s < D; ++s)
#pragma unroll
    for (int j = 0; j < TY; ++j) load_d(s, j);
  __builtin_amdgcn_sched_barrier(0);
  auto period = [&](auto last) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const bool fetch = !decltype(last)::value || s + D < P;
      v4i y[TY];
#pragma unroll
      for (int j = 0; j < TY; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) y[j][d] = yf[s % D][j][d] ^ (int)0x80808080;
#pragma unroll
      for (int i = 0; i < TX; ++i) {
#pragma unroll
        for (int j = 0; j < TY; ++j) {
          acc[i][j] = OpI8::mma(xf[s % D][i], y[j], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
          if (fetch && i == 0) load_d(s + D, j);
          if (fetch && j == TY - 1)
            xf[s % D][i] = __builtin_bit_cast(
                v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + sw + (u32)(s + D) * 1024u), 0));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  for (int s = s0; s + P < s1; s += P) {
    period(std::false_type{});
    soff += 2 * hw16;
    sw += P * 1024u;
  }
  period(std::true_type{});
}

// requant_row's arithmetic for four channels, the addend already in them
__device__ __forceinline__ int requant_quad(const v4i &v, int scale, int shift) {
  if (shift >= 33) {
    const int rhi = 1 << (shift - 33), sh = shift - 32;
    const u32 lo = (unsigned short)__builtin_amdgcn_ashr_pk_u8_i32(__mulhi(v[0], scale) + rhi, __mulhi(v[1], scale) + rhi, sh);
    const u32 hi = (unsigned short)__builtin_amdgcn_ashr_pk_u8_i32(__mulhi(v[2], scale) + rhi, __mulhi(v[3], scale) + rhi, sh);
    return (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
  }
  u32 packed = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const long long t = ((long long)v[e] * scale + (1ll << (shift - 1))) >> shift;
    packed |= (u32)(t < 0 ? 0 : (t > 255 ? 255 : t)) << (8 * e);
  }
  return (int)packed;
}

// MODE 4: 3 x 3 windows at stride 1 whose output is as large as their input, and a share of whole periods: the pixels under a
// wave's windows are a run of 32 TY + 2 W + 2 pixels per channel block, delivered once into the wave's own part of LDS instead of
// up to nine times into registers: a 64 x 64 tile on 14 x 14 takes 8 KiB of pixels, not 36.  Raw buffer loads: what lies
// outside the group arrives as zeros, and so does the last pixel of a block's rows, which stands for padding.  us with MODE 3 /
// here: ResNet-50 batch 1 152 / 150, 16 244 / 237, 32 362 / 350; ResNet-18 64 / 62, 82 / 79, 109 - 113 / 102 - 110 (machine to
// machine).  Weights nine steps ahead for 64 x 64 tiles spill (batch 32 369), and so do whole steps unrolled (146 registers);
// staged through registers, exclusive-ors done there, 357.
template <int TX, int TY> constexpr int kRingPatch = TX * TY == 4 ? 3 : 9;
__host__ __device__ constexpr int patch_rows(int pixels, int w) { return (pixels + 2 * w + 2) / 64 + 1; }  // of 64 pixels, 1 KiB
template <int TX, int TY>
__device__ __forceinline__ void chain_reduce_patch(v16i (&acc)[TX][TY], __amdgpu_buffer_rsrc_t wbuf, const u32 (&wp)[TX], const u32 lane16,
                                                   const char *patch, const u32 (&inside)[TY], v4i (&xf)[kMaxRing<TX, TY>][TX], int half,
                                                   int s0, int s1, int rows, int w16) {
  constexpr int P = 9, D = kRingPatch<TX, TY>, Y = 3;
  static_assert(P % D == 0 && P % Y == 0 && D <= kMaxRing<TX, TY>, "the rings' slots repeat with the period");
  const u32 l16 = lane16 & 511u, padding = (u32)(rows * 1024 - 16);
  u32 at[P][TY];  // tap 2 s + half of a period
#pragma unroll
  for (int s = 0; s < P; ++s) {
    const int e = 2 * s, o = 2 * s + 1;
    const u32 oe = (u32)((e / 9) * rows * 1024 + (e % 9 / 3) * w16 + (e % 9 % 3) * 16);
    const u32 oo = (u32)((o / 9) * rows * 1024 + (o % 9 / 3) * w16 + (o % 9 % 3) * 16);
#pragma unroll
    for (int j = 0; j < TY; ++j)
      at[s][j] = inside[j] >> (half ? o % 9 : e % 9) & 1u ? l16 + (u32)(j * 512) + (half ? oo : oe) : padding;
  }
  v4i yf[Y][TY];
  auto load_d = [&](int s, int j) __attribute__((always_inline)) {
    yf[s % Y][j] = *reinterpret_cast<const v4i *>(patch + at[s % P][j] + (u32)(s / P * 2 * rows * 1024));
  };
#pragma unroll
  for (int s = 0; s < Y; ++s)
#pragma unroll
    for (int j = 0; j < TY; ++j) load_d(s, j);
  u32 sw = (u32)(s0 + D) * 1024u;
  auto period = [&](auto last) __attribute__((always_inline)) {
    constexpr bool kLast = decltype(last)::value;
#pragma unroll
    for (int s = 0; s < P; ++s) {
      v4i y[TY];
#pragma unroll
      for (int j = 0; j < TY; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) y[j][d] = yf[s % Y][j][d] ^ (int)0x80808080;
#pragma unroll
      for (int i = 0; i < TX; ++i) {
#pragma unroll
        for (int j = 0; j < TY; ++j) {
          acc[i][j] = OpI8::mma(xf[s % D][i], y[j], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0 && (!kLast || s + Y < P)) load_d(s + Y, j);
          if (j == TY - 1 && (!kLast || s + D < P))
            xf[s % D][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + sw + (u32)s * 1024u), 0));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  for (int s = s0; s + P < s1; s += P) {
    period(std::false_type{});
    patch += 2 * rows * 1024;
    sw += P * 1024u;
  }
  period(std::true_type{});
}

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kPerCu, kPerCu))) void chain_run(const ChainArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  ChainLds &sh = *reinterpret_cast<ChainLds *>(lds_raw);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = __builtin_amdgcn_s_getreg((31 << 11) | 20) & (kMaxXcd - 1);
  const StepPtr steps = (StepPtr)(unsigned long long)a.steps;
  int *const tickets = a.ctl + kCtlTickets + 32 * xcd;
  int *const slots = a.ctl + kCtlSlots + xcd * a.slot_pitch;
  if (tid == 0) sh.ticket[0] = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  int turn = 0, q_now = -1, group = 0, l = 0, budget = a.polls;
  for (;;) {
    const int ticket = __builtin_amdgcn_readfirstlane(sh.ticket[turn]);
    turn ^= 1;
    int q, idx;
    a.by_tickets.divmod(ticket, q, idx);
    if (q != q_now) {
      if (q >= a.groups) break;
      if (tid == 0) {
        int v;
        if (idx == 0) {
          v = __hip_atomic_fetch_add(a.ctl + kCtlGroups, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
          store_result<0>(result_buffer(slots), (u32)q * 4u, v);
        } else {
          while ((v = load_l2(slots + q)) == 0 && --budget > 0) __builtin_amdgcn_s_sleep(1);
          if (v == 0) v = a.groups + 1;
        }
        sh.group = v - 1;
      }
      __syncthreads();
      group = __builtin_amdgcn_readfirstlane(sh.group);
      q_now = q;
      l = 0;
    }
    if (group >= a.groups) break;
    ChainStep L = load_step(steps + l);
    while (idx >= L.next) L = load_step(steps + ++l);
    const int nct = L.nct, ohw = L.ohw, K = L.K, nsteps = L.nsteps, kl = L.kg_log, wl = L.wx_log;
    const int local = idx - L.first;
    const int pt = quot(local, L.by_nct), ct = local - pt * nct;
    const int image0 = group * a.per, npix = min(a.per, a.images - image0) * ohw;
    const int tx = L.tile & 15, ty = L.tile >> 4, m0 = pt << (ty + L.wy_log), me = min(m0 + (1 << (ty + L.wy_log)), npix) - 1;
    if (m0 > me) {  // the last group may hold fewer images
      if (tid == 0) sh.ticket[turn] = __hip_atomic_fetch_add(tickets, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      continue;
    }
    const int set = wave >> kl, kidx = wave & ((1 << kl) - 1);
    const int x0 = ((ct << wl) + (set & ((1 << wl) - 1))) << tx, y0 = m0 + ((set >> wl) << ty);
    const bool idle = x0 >= K || y0 >= npix;
    const int s0 = idle ? 0 : (nsteps * kidx) >> kl, s1 = idle ? 0 : (nsteps * (kidx + 1)) >> kl;
    const int slast = max(s1 - 1, s0);

    // the source layer's tiles that this one reads: their flags are asked for first and looked at when the loads of
    // the weights are out
    const int H = L.H, W = L.W;
    int lo = m0, hi = me;
    if (!L.flat) {
      const int n0 = quot(m0, L.by_ohw), n1 = quot(me, L.by_ohw), hw = H * W;
      const int r0 = quot(m0 - n0 * ohw, L.by_ow) * L.sh - L.pt;
      const int r1 = quot(me - n1 * ohw, L.by_ow) * L.sh - L.pt + L.KH - 1;
      lo = n0 * hw + min(max(r0, 0), H - 1) * W;
      hi = n1 * hw + max(min(r1, H - 1), 0) * W + W - 1;
    }
    int *const flags = a.ctl + (size_t)(u32)(a.flags0 + group * a.flag_pitch);
    const int *const wanted = flags + L.src_first;
    const int fa = (lo >> L.src_shift) * L.src_nct, fb = ((hi >> L.src_shift) + 1) * L.src_nct;
    const int flag = load_l2(wanted + (u32)min(fa + lane, max(fb - 1, 0)));
    __builtin_amdgcn_sched_barrier(0);

    int next = 0;
    auto tile = [&](auto tx_, auto ty_) __attribute__((always_inline)) {
      constexpr int TX = decltype(tx_)::value, TY = decltype(ty_)::value;
      // weights: the ring's fragments depend on the tile alone
      const u32 lane16 = (u32)lane * 16u;
      const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc((void *)L.w, 0, -1, 0x00020000);
      const int kblocks = (K + 31) >> 5;
      u32 wp[TX];  // byte offsets of the 32-channel blocks; blocks past the last one re-read it
#pragma unroll
      for (int i = 0; i < TX; ++i) wp[i] = (u32)(min((x0 >> 5) + i, kblocks - 1) * nsteps) * 1024u;
      v4i xf[kMaxRing<TX, TY>][TX];
      auto load_w = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TX; ++i)
          xf[u][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, (int)lane16, (int)(wp[i] + (u32)min(s0 + u, slast) * 1024u), 0));
      };
#pragma unroll
      for (int u = 0; u < kShort<TX, TY>; ++u) load_w(u);
      const bool is_short = s1 - s0 <= kShort<TX, TY> && L.mode == 0;
      if (!is_short) {
#pragma unroll
        for (int u = kShort<TX, TY>; u < kRing<TX, TY>; ++u) load_w(u);
        if (kRing<TX, TY> < kRingPatch<TX, TY> && L.mode == 4) {
#pragma unroll
          for (int u = kRing<TX, TY>; u < kRingPatch<TX, TY>; ++u) load_w(u);
        }
      }
      const u32 cc = (u32)min(x0 + lane, K - 1) * 4u;
      const int add0 = __builtin_amdgcn_raw_buffer_load_b32(wbuf, (int)cc, kblocks * nsteps * 1024, 0);
      const int add1 = L.bias ? ((Global<int>)L.bias)[cc >> 2] : 0;
      __builtin_amdgcn_sched_barrier(0);

      const __amdgpu_buffer_rsrc_t data = __builtin_amdgcn_make_buffer_rsrc(
          (void *)(L.data + (size_t)image0 * (size_t)(u32)L.img_bytes), 0, min(a.per, a.images - image0) * L.img_bytes, 0x00020000);
      int pixoff[TY];
      u32 inside[TY], dst[TY];
#pragma unroll
      for (int j = 0; j < TY; ++j) {
        const int m = y0 + j * 32 + l32;
        const int mm = m < npix ? m : 0;
        const int n = quot(mm, L.by_ohw), pix = mm - n * ohw;
        dst[j] = ((u32)(n * (K >> 4) * ohw) + (u32)pix) * 16u;
        inside[j] = 0;
        if (L.flat) {
          pixoff[j] = n * L.img_bytes + pix * 16;
        } else {
          const int oh = quot(pix, L.by_ow), ow = pix - __mul24(oh, (int)L.OW);
          const int ih0 = __mul24(oh, (int)L.sh) - L.pt, iw0 = __mul24(ow, (int)L.sw) - L.pl;
          pixoff[j] = n * L.img_bytes + (__mul24(ih0, W) + iw0) * 16;
          if (L.mode >= 2) {
            const int KH = L.KH, KW = L.KW;
            const int ka = min(max(-iw0, 0), KW), kb = min(max(W - iw0, ka), KW);
            const int ra = min(max(-ih0, 0), KH), rb = min(max(H - ih0, ra), KH);
            const u32 rows = L.row_ones & ((1u << __mul24(rb, KW)) - (1u << __mul24(ra, KW)));
            inside[j] = m < npix ? ((1u << kb) - (1u << ka)) * rows : 0u;
          }
        }
      }
      if (L.reads) {
        if (!__all(flag != 0))
          while (!__all(load_l2(wanted + (u32)min(fa + lane, fb - 1)) != 0) && --budget > 0) __builtin_amdgcn_s_sleep(1);
        for (int b = fa + 64; b < fb; b += 64) {
          while (!__all(load_l2(wanted + (u32)min(b + lane, fb - 1)) != 0) && --budget > 0) __builtin_amdgcn_s_sleep(1);
        }
      }

      v16i acc[TX][TY];
#pragma unroll
      for (int i = 0; i < TX; ++i)
#pragma unroll
        for (int j = 0; j < TY; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
      const TapWalk tw{L.ntaps, L.KW, L.win, (W - L.KW) * 16, (H - L.KH) * W * 16, H * W * 16, W * 16, L.by_win, L.by_kw};
      if (L.mode == 4) {
        if (s0 < s1) {
          const int rows = patch_rows(32 * TY, W), cb0 = 2 * (s0 / 9), cb1 = 2 * (s1 / 9);
          char *const patch = reinterpret_cast<char *>(sh.part[wave]);
          for (int k = 0; k < rows; ++k) {
            const int p = k * 64 + lane, m = y0 - W - 1 + p;
            const int n = quot(max(m, 0), L.by_ohw);
            const u32 from = m >= 0 && m < npix && p < rows * 64 - 1 ? (u32)(n * L.img_bytes + (m - n * ohw) * 16) : ~0u;
            for (int cb = cb0; cb < cb1; ++cb)
              __builtin_amdgcn_raw_ptr_buffer_load_lds(data, (__attribute__((address_space(3))) void *)(patch + ((cb - cb0) * rows + k) * 1024), 16, (int)from, cb * ohw * 16, 0, kAgent);
          }
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
          chain_reduce_patch<TX, TY>(acc, wbuf, wp, lane16, patch, inside, xf, half, s0, s1, rows, W * 16);
        }
      } else if (L.mode == 3) {
        if (s0 < s1) chain_reduce_3x3<TX, TY>(acc, wbuf, wp, data, lane16, pixoff, inside, xf, half, s0, s1, H * W * 16, W * 16);
      } else if (is_short)
        chain_reduce<0, TX, TY, kShort<TX, TY>, true>(acc, wbuf, wp, data, lane16, pixoff, inside, xf, half, s0, s1, slast, tw);
      else if (L.mode == 0)
        chain_reduce<0, TX, TY, kRing<TX, TY>, false>(acc, wbuf, wp, data, lane16, pixoff, inside, xf, half, s0, s1, slast, tw);
      else if (L.mode == 1)
        chain_reduce<1, TX, TY, kRing<TX, TY>, false>(acc, wbuf, wp, data, lane16, pixoff, inside, xf, half, s0, s1, slast, tw);
      else
        chain_reduce<2, TX, TY, kRing<TX, TY>, false>(acc, wbuf, wp, data, lane16, pixoff, inside, xf, half, s0, s1, slast, tw);
      // Taken no earlier: a workgroup that still waits would tie a later tile to itself (a tile earlier: 151 -> 161 us at batch 1)
      sh.addend[wave][lane] = add0 + add1;
      __builtin_amdgcn_sched_barrier(0);
      if (tid == 0) {
        // divergent as far as the compiler knows: of a uniform address it makes a wave-wide sum, and waits for it on the spot, 0.3 us
        // a tile (batch 1 164 / 154 us, batch 32 376 / 366)
        auto *at = (__attribute__((address_space(1))) int *)tickets;
        asm("" : "+v"(at));
        next = __hip_atomic_fetch_add(at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      const __amdgpu_buffer_rsrc_t obuf = result_buffer(L.out + (size_t)image0 * (size_t)(u32)(K * ohw));
      auto store = [&](int i, int j, const v16i &v) __attribute__((always_inline)) {
        const v4i row = requant_row(v, &sh.addend[wave][i * 32], L.scale, L.shift, half);
        const int c = x0 + i * 32 + half * 16;
        if (c < K && y0 + j * 32 + l32 < npix) store_result<0>(obuf, dst[j] + (u32)((c >> 4) * ohw) * 16u, row);
      };
      // KG k-groups: each parks the quads (four channels of a lane's pixel) that others own and adds up its own
      auto finish = [&](auto kg_) __attribute__((always_inline)) {
        constexpr int KG = decltype(kg_)::value, QUADS = 4 * TX * TY, OWN = QUADS / KG;
        auto quad = [&](int q) __attribute__((always_inline)) {
          const v16i &v = acc[q / 4 / TY][q / 4 % TY];
          return v4i{v[4 * (q & 3)], v[4 * (q & 3) + 1], v[4 * (q & 3) + 2], v[4 * (q & 3) + 3]};
        };
        auto sum = [&](int q) __attribute__((always_inline)) {
          v4i v = quad(q);
#pragma unroll
          for (int o = 1; o < KG; ++o) v += sh.part[set * KG + ((kidx + o) & (KG - 1))][q][lane];
          return v;
        };
#pragma unroll
        for (int o = 0; o < KG; ++o)
          if (o != kidx) {
#pragma unroll
            for (int q = o * OWN; q < (o + 1) * OWN; ++q) sh.part[wave][q][lane] = quad(q);
          }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < KG; ++o)
          if (o == kidx) {
            if constexpr (OWN % 4 == 0) {
#pragma unroll
              for (int b = o * OWN / 4; b < (o + 1) * OWN / 4; ++b) {
                v16i v;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const v4i x = sum(4 * b + q);
#pragma unroll
                  for (int e = 0; e < 4; ++e) v[4 * q + e] = x[e];
                }
                store(b / TY, b % TY, v);
              }
            } else {
#pragma unroll
              for (int q = o * OWN; q < (o + 1) * OWN; ++q) {
                const int i = q / 4 / TY, j = q / 4 % TY, c = x0 + i * 32 + (q >> 1 & 1) * 16;
                const v4i v = sum(q) + *reinterpret_cast<const v4i *>(&sh.addend[wave][i * 32 + 8 * (q & 3) + 4 * half]);
                if (c < K && y0 + j * 32 + l32 < npix)
                  store_result<0>(obuf, dst[j] + (u32)((c >> 4) * ohw) * 16u + (u32)((q & 1) * 8 + half * 4), requant_quad(v, L.scale, L.shift));
              }
            }
          }
      };
      if (kl == 2) {
        finish(std::integral_constant<int, 4>{});
      } else if (kl == 1) {
        finish(std::integral_constant<int, 2>{});
      } else {
#pragma unroll
        for (int b = 0; b < TX * TY; ++b) store(b / TY, b % TY, acc[b / TY][b % TY]);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // results are in this XCD's L2
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    if (ty == 6)
      tile(Two{}, Two{});
    else if (tx == 6)
      tile(Two{}, One{});
    else
      tile(One{}, One{});
    if (tid == 0) sh.ticket[turn] = next;
    __syncthreads();
    if (tid == 0) store_result<0>(result_buffer(flags), (u32)idx * 4u, 1);
  }
  if (budget <= 0) give_up(a);  // here and not at the waits: a store there cost every run 2 - 10 us
}

struct ChainPlan {
  int per, groups, tickets, slot_pitch, flags0, flag_pitch, clear_words;
  size_t steps_off, bytes;
};

struct Rings {  // k-steps in flight
  int of_walk, of_short, of_3x3, of_patch;
};
template <int TX, int TY>
constexpr Rings rings() {
  return {kRing<TX, TY>, kShort<TX, TY>, kRing3<TX, TY>, kRingPatch<TX, TY>};
}

struct Range {
  const char *a, *b;
};

// Every run makes its plan again, so sizes of tiles and k-groups, powers of two, stand here as their logarithms (shifts, no
// divisions), and what few chains need (estimate64) is worked out for those: ResNet-50 5.8 us of host time, 10.6 without either.
inline long ceil_shift(long n, int log) { return (n + (1l << log) - 1) >> log; }

// the reduction (MODE) of a layer in 1 << klog k-groups: all of them at once, one for each tile height of 32 and 64 pixels
struct Modes {
  unsigned char of[2][3];
  Modes(const unit_conv_desc &d, const ChainStep &s) {
    const int ntaps = s.ntaps, W = d.W;
    const int plain = d.pt || d.pl || d.pb || d.pr ? 2 : d.KH * d.KW == 1 && ntaps % 2 == 0 ? 0 : 1;
    const int periods = d.KH == 3 && d.KW == 3 && ntaps % 18 == 0 ? ntaps / 18 : 0;  // of nine k-steps
    const bool same = d.sh == 1 && d.sw == 1 && d.pt == 1 && d.pl == 1 && s.OW == W && s.ohw == d.H * W;
    for (int y = 0; y < 2; ++y)
      for (int k = 0; k < 3; ++k) {
        // a wave's part of LDS is 16 KiB
        const bool fits = same && (d.C >> (4 + k)) * patch_rows(32 << y, W) <= (int)sizeof(ChainLds::part) / kWaves / 1024;
        of[y][k] = (unsigned char)(!periods || periods & ((1 << k) - 1) ? plain : fits ? 4 : 3);
      }
  }
};

// rounds of an XCD's 64 workgroups; x: log2 of a workgroup's waves side by side along the channels
inline double rounds_of(int K, long npix, int xlog, int ylog, int klog, int &x) {
  x = std::max(0, std::min(2 - klog, 31 - __builtin_clz((u32)K) - xlog));
  return (double)(ceil_shift(K, xlog + x) * ceil_shift(npix, ylog + 2 - klog - x)) * 0.015625;
}

// us of all layers on 64 x 64 tiles alone
inline double estimate64(const unit_chain_layer *layers, const ChainStep *st, int count, int per) {
  double here = 5.5;
  for (int i = 0; i < count; ++i) {
    const ChainStep &s = st[i];
    const long npix = (long)per * s.ohw;
    int kg = 0, x;
    double best = 1e30;
    const double tiles = (double)(ceil_shift(s.K, 6) * ceil_shift(npix, 6));
    for (int k = 0; k <= 2 && 1 << k <= s.nsteps; ++k) {
      const double t = std::max(1.0, tiles * (1 << k) * 0.00390625) * (2.6 + (k ? 0.4 : 0.0) + 0.25 * ceil_shift(s.nsteps, k));
      if (t < best) best = t, kg = k;
    }
    const double rounds = rounds_of(s.K, npix, 6, 6, kg, x), mb = 1e-6 * ((double)(u32)s.img_bytes + (double)s.ohw * s.K);
    const int mode = Modes(layers[i].desc, s).of[1][kg];
    here += 1.45 + (kg ? 0.15 : 0.0) + 0.8 * std::max(1.0, rounds) +
            (mode == 1 || mode == 2 ? 0.3 : 0.21) * ceil_shift(s.nsteps, kg) * std::max(0.5, rounds) + 1.28 * mb * per;
  }
  return here;
}

// false: the layers run one launch each
bool plan_chain(const unit_chain_layer *layers, int count, const void *x, ChainStep *st, ChainPlan *p) {
  if (count < 2 || count > kMaxChain) return false;
  const int N = layers[0].desc.N;
  if (N < 1) return false;
  // one group per XCD (smaller ones, two in a row: batch 64 773 against 621 us; larger ones leave XCDs idle)
  const int per = (N + 7) / 8;
  p->per = per;
  p->groups = (N + per - 1) / per;
  long first = 0;
  double here = 5.35, launches = 0.9;  // us, below
  Range outs[kMaxChain];
  for (int i = 0; i < count; ++i) {
    const unit_chain_layer &l = layers[i];
    const unit_conv_desc &d = l.desc;
    if (!l.prepared || !l.out || l.shift < 1 || l.shift > 62 || check_aligned("chain", {l.data, l.prepared, l.out})) return false;
    if (d.N != N || d.cb != 16 || d.dh != 1 || d.dw != 1 || d.C <= 0 || d.K <= 0 || d.KH <= 0 || d.KW <= 0) return false;
    ConvGeom g;
    if (conv_sizes(&d, 16, &g, "chain") != UNIT_OK) return false;
    if (d.KH * d.KW > 31 || d.sh > 255 || d.sw > 255 || d.pt > 255 || d.pl > 255) return false;
    const long out_bytes = (long)g.npix * d.K;
    if (out_bytes > 0x7fffffffl) return false;
    outs[i] = Range{static_cast<const char *>(l.out), static_cast<const char *>(l.out) + out_bytes};
    ChainStep &s = st[i];
    s.data = static_cast<const char *>(l.data ? l.data : x);
    s.w = static_cast<const char *>(l.prepared);
    s.out = static_cast<char *>(l.out);
    s.bias = l.bias;
    // doubled up to a shift of 33, while there is room for the sign
    const int up = std::max(0, std::min(33 - l.shift, l.scale ? __builtin_clrsb(l.scale) : 32));
    s.scale = (int)((unsigned long long)(u32)l.scale << up);
    s.shift = (unsigned char)(l.shift + up);
    s.K = d.K;
    s.ntaps = g.ntaps;
    s.nsteps = (g.ntaps + 1) / 2;
    s.ohw = g.OH * g.OW;
    s.win = (unsigned char)(d.KH * d.KW);
    s.img_bytes = (int)g.img_bytes;
    s.by_ohw = small_div(s.ohw);
    s.by_ow = small_div(g.OW);
    s.by_win = small_div(s.win);
    s.by_kw = small_div(d.KW);
    s.H = (unsigned short)d.H, s.W = (unsigned short)d.W, s.OW = (unsigned short)g.OW;
    s.pt = (unsigned char)d.pt, s.pl = (unsigned char)d.pl;
    s.row_ones = g.row_ones;
    s.KH = (unsigned char)d.KH, s.KW = (unsigned char)d.KW, s.sh = (unsigned char)d.sh, s.sw = (unsigned char)d.sw;
    const bool masked = d.pt || d.pl || d.pb || d.pr;
    s.flat = !masked && d.KH == 1 && d.KW == 1 && d.sh == 1 && d.sw == 1;
    const long npix = (long)per * s.ohw;
    if (npix * s.ohw > 0x7fffffffl) return false;
    // Tile and k-groups.  A layer costs the decode, first loads, requantisation, stores and flag of its tiles (2.1 - 2.5 us, 0.1 more
    // with k-groups, 1.9 for each further round of an XCD's 64 workgroups) and a price per k-step of a wave: by tile and walk, less while
    // workgroups are idle, since the others then have the loads to themselves.  Smaller tiles move more operand bytes per result and
    // pay where large ones leave workgroups idle; k-groups that leave whole periods of nine k-steps keep the cheap walk (3 x 3, 64
    // channels, 28 x 28, batch 4: four groups of 5 k-steps that walk 3.8 us a layer, two of 9 2.7).  Fitted to 1400 chains of two
    // alternating layers, each with all nine combinations, but for 1 x 1 layers on 32 x 32 tiles: 0.10 by the fit, with which ResNet-50 at
    // 12 images and more is 3 - 10 % slower (what its layers have that those chains lack is not in these prices).  The choice is 2.0 %
    // from the best one (geometric mean).  us with 64 x 64 alone / now: ResNet-50 batch 1 203 / 151, 8 232 / 171, 16 275 / 237,
    // 32 377 / 350; ResNet-18 1 83 / 62, 32 118 / 110; 1309 random chains 1.23 in the mean, seven of them 3 - 9 % slower, and 59 of
    // the 1400: mostly tiles of few k-steps that occupy every workgroup (1 x 1 128 -> 128 on 32 x 32, two images, 16 layers 42.5 / 47.2; 3 x 3
    // 112 -> 112 on 32 x 32, eight images, six layers 40.3 / 44.7), one with weights beyond the L2 (3 x 3 256 - 2048 on 14 x 14, eight
    // images, 276 / 372).  0.5 us more from half a round to a full one, refitted: random chains 1.01, ResNet-50 at up to eight images 3 -
    // 4 % slower; 0.2 us, not for 1 x 1 layers: 78 of 1200 random chains gain more than 3 %, five lose up to 9.  Neither is taken.
    const Modes modes(d, s);
    const int K = d.K, nsteps = s.nsteps;
    int kg = 0, sx = 6, sy = 6, wx = 0;
    double tiles_us = 1e30, steps_us = 0;
    const auto offer = [&](int xlog, int ylog, double first, const double (&step)[5]) {
      for (int k = 0; k <= 2 && 1 << k <= nsteps; ++k) {
        int x;
        const double rounds = rounds_of(K, npix, xlog, ylog, k, x);
        const double t = first + (k ? 0.1 : 0.0) + 1.9 * std::max(0.0, rounds - 1);
        const double u = step[modes.of[ylog - 5][k]] * ceil_shift(nsteps, k) * std::max(rounds, 0.5 + 0.5 * std::min(1.0, rounds));
        if (t + u < tiles_us + steps_us) tiles_us = t, steps_us = u, kg = k, sx = xlog, sy = ylog, wx = x;
      }
    };
    offer(6, 6, 2.5, {0.27, 0.32, 0.32, 0.26, 0.24});
    offer(6, 5, 2.15, {0.2, 0.26, 0.26, 0.19, 0.15});
    offer(5, 5, 2.1, {0.15, 0.21, 0.21, 0.12, 0.09});
    s.mode = modes.of[sy - 5][kg];
    const int wy = 2 - kg - wx, cols = sx + wx, rows = sy + wy;
    s.kg_log = (unsigned char)kg, s.wx_log = (unsigned char)wx, s.wy_log = (unsigned char)wy;
    s.tile = (unsigned char)(sx | sy << 4);
    s.nct = (int)ceil_shift(K, cols);
    s.by_nct = small_div(s.nct);
    const long npt = ceil_shift(npix, rows);
    if (npt * s.nct * s.nct > 0x7fffffffl) return false;
    const double gmac = 1e-9 * s.ohw * d.K * s.ntaps * 16, mb = 1e-6 * ((double)g.img_bytes + (double)s.ohw * d.K);  // of an image
    here += 0.78 * tiles_us + 1.06 * steps_us + 0.9 * mb * per;
    launches += 3.6 + 1.15 * gmac * N + 0.176 * mb * N + 0.019 * std::min(s.nsteps, 80);
    s.first = (int)first;
    first += npt * s.nct;
    s.next = (int)first;
    if (first * (p->groups + 2) + 4096 > 0x7fffffffl) return false;
    s.reads = 0, s.src_first = 0, s.src_nct = 0, s.src_shift = 0;
    for (int j = i - 1; j >= 0; --j)
      if (layers[j].out == s.data) {
        if (layers[j].desc.K != d.C || st[j].OW != d.W || st[j].ohw != d.H * d.W) return false;
        s.reads = 1;
        s.src_first = st[j].first, s.src_nct = st[j].nct, s.src_shift = (unsigned char)((st[j].tile >> 4) + st[j].wy_log);
        break;
      }
  }
  // Short chains, few images through large layers and activations that outgrow an XCD's 4 MB of L2 stay launches.  The kernel
  // costs 5.4 us before its first tile, then the layers as estimated above and 0.9 us per MB that the group reads and writes; a launch
  // 3.6 us, 1.2 per GMAC and 0.18 per MB of the batch.  estimate64 is the one for 64 x 64 tiles alone (a layer 1.5 us, 0.8 for each
  // round of an XCD's 64 workgroups, 0.2, with the tap walk 0.3, per k-step of it); the tiles taken are 1.23 times as fast in the mean, but
  // no chain is sure to be (above).  Both have errors of 6 - 7 % (root mean square) that differ, and either one is taken at its word, for
  // what that measured: over 500 random chains of 3 to 48 layers
  // timed both ways, estimate64 alone ends 2.4 % from always the faster way, `here` alone 1.2 %, either 0.8 %; of the 413 given to
  // the kernel two lose more than 3 % there, both of 3 layers.  us here / as launches: 3 x 3 64 -> 64 on 56 x 56, batch 8, 3 layers
  // 17.6 / 20.1; 1 x 1 256 -> 256 on 14 x 14, batch 1, 8 layers 24.3 / 30.3; the other way, with 64 x 64 tiles, 14 layers from
  // 51 x 51, batch 14 245 / 201, 10 layers from 50 x 50, batch 52 197 / 167, 9 layers of 224 channels on 20 x 20, batch 2 42.9 / 38.0.
  if (here > 0.93 * launches && estimate64(layers, st, count, per) > 0.975 * launches) return false;
  // The layers no longer run one after the other: none may write what another one reads or writes, but for a source's
  // whole result.
  std::sort(outs, outs + count, [](const Range &u, const Range &v) { return u.a < v.a; });
  for (int i = 1; i < count; ++i)
    if (outs[i].a < outs[i - 1].b) return false;
  const auto clear_of_outs = [&](const void *q, size_t n) {
    const char *a = static_cast<const char *>(q), *b = a + n;
    const Range *r = std::upper_bound(outs, outs + count, a, [](const char *v, const Range &u) { return v < u.b; });
    return r == outs + count || r->a >= b;
  };
  for (int i = 0; i < count; ++i) {
    const unit_conv_desc &d = layers[i].desc;
    if (!clear_of_outs(st[i].w, prepared_layout(d.K, d.C, d.KH, d.KW, 16, 1).total_bytes)) return false;
    if (st[i].bias && !clear_of_outs(st[i].bias, (size_t)d.K * 4)) return false;
    if (!st[i].reads && !clear_of_outs(st[i].data, (size_t)N * d.C * d.H * d.W)) return false;
  }
  p->tickets = (int)first;
  p->slot_pitch = (p->groups + 31) / 32 * 32;
  p->flags0 = kCtlSlots + kMaxXcd * p->slot_pitch;
  p->flag_pitch = (p->tickets + 31) / 32 * 32;
  p->clear_words = p->flags0 + p->groups * p->flag_pitch;
  p->steps_off = ((size_t)p->clear_words * 4 + 255) / 256 * 256;
  p->bytes = p->steps_off + (size_t)(count + 1) * sizeof(ChainStep) + kWsAlign;  // ws itself is at 16 bytes, and its head in front
  return true;
}

}  // namespace
}  // namespace unit

extern "C" int unit_conv_chain_u8_ws_bytes(const unit_chain_layer *layers, int32_t count, size_t *bytes) {
  using namespace unit;
  if (!layers || !bytes || count < 0) return fail(UNIT_E_ARG, "unit_conv_chain_u8_ws_bytes: null pointer or negative count");
  ChainStep st[kMaxChain];
  ChainPlan p;
  *bytes = plan_chain(layers, count, nullptr, st, &p) ? p.bytes : 0;
  return UNIT_OK;
}

extern "C" int unit_conv_chain_u8_ws(const unit_chain_layer *layers, int32_t count, const void *x, void *ws, size_t ws_bytes,
                                     unit_stream_t stream) {
  return unit_conv_chain_u8_status(layers, count, x, ws, ws_bytes, nullptr, stream);
}

extern "C" int unit_conv_chain_u8_status(const unit_chain_layer *layers, int32_t count, const void *x, void *ws, size_t ws_bytes,
                                         int32_t *status, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_conv_chain_u8_ws";
  if (!layers || !x || count < 0) return fail(UNIT_E_ARG, "%s: null pointer or negative count", what);
  if (reinterpret_cast<uintptr_t>(status) % 4) return fail(UNIT_E_ARG, "%s: status must be 4-byte aligned", what);
  ChainStep st[kMaxChain];
  ChainPlan p;
  const bool pinned = tuning_override("UNIT_AMD_CONV_VARIANT") > 0 || tuning_override("UNIT_AMD_CONV_PANEL") > 0 ||
                      tuning_override("UNIT_AMD_CONV_SPLITK") > 0;
  if (!ws || reinterpret_cast<uintptr_t>(ws) % 16 || reinterpret_cast<uintptr_t>(x) % 16 || pinned ||
      !plan_chain(layers, count, x, st, &p) || ws_bytes < p.bytes)
    return unit_conv_chain_u8(layers, count, x, stream);
  if (int rc = check_device()) return rc;
  static thread_local bool allowed = false;  // the opt-in for > 64 KiB of dynamic LDS is sticky per kernel
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(chain_run), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    allowed = true;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  char *base = reinterpret_cast<char *>((reinterpret_cast<uintptr_t>(ws) + kWsHead + kWsAlign - 1) / kWsAlign * kWsAlign);
  ChainStep *steps = reinterpret_cast<ChainStep *>(base + p.steps_off);
  for (int i = 0; i <= count; i += kSetupSteps) {  // the status word's entry, then the layers
    ChainSetup a;
    const int n = std::min(kSetupSteps, count + 1 - i), head = i == 0;
    if (head) {
      memset(a.s, 0, sizeof(ChainStep));
      a.s[0].out = reinterpret_cast<char *>(status ? status : static_cast<int32_t *>(ws));
    }
    memcpy(a.s + head, st + i - !head, (n - head) * sizeof(ChainStep));
    const int quads = i == 0 ? ceil_div(p.clear_words, 4) : 0;
    hipLaunchKernelGGL(chain_setup, dim3(std::max(1, std::min(256, ceil_div(quads, 256)))), dim3(256), 0, s, a, steps + i, n,
                       reinterpret_cast<v4i *>(base), quads);
  }
  const int polls = tuning_override("UNIT_AMD_CHAIN_POLLS");
  const ChainArgs a{steps + 1, reinterpret_cast<int *>(base), polls > 0 ? polls : kPolls, layers[0].desc.N, p.per, p.groups,
                    p.slot_pitch, p.flags0, p.flag_pitch, FastDiv::make(p.tickets)};
  hipLaunchKernelGGL(chain_run, dim3(256 * kPerCu), dim3(kThreads), sizeof(ChainLds), s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
  // the workgroup's tile, its k-groups, the k-steps in flight of the general walk (5, 6, 9: wave tiles of 64 x 64, 64 x 32, 32 x 32),
  // the layer's own walk (MODE) and the k-steps of weights in flight in that
  for (int i = 0; i < count; ++i)
    if (layers[i].variant) {
      const ChainStep &t = st[i];
      const Rings r = t.tile >> 4 == 6 ? rings<2, 2>() : (t.tile & 15) == 6 ? rings<2, 1>() : rings<1, 1>();
      const bool is_short = t.mode == 0 && ceil_shift(t.nsteps, t.kg_log) <= r.of_short;
      snprintf(layers[i].variant, 96, "q8chain_x%d_y%d_g%d_d%d_m%d_r%d", 1 << ((t.tile & 15) + t.wx_log), 1 << ((t.tile >> 4) + t.wy_log),
               1 << t.kg_log, r.of_walk, t.mode, is_short ? r.of_short : t.mode == 4 ? r.of_patch : t.mode == 3 ? r.of_3x3 : r.of_walk);
    }
  set_variant("q8chain_l%d_n%d_d%d", count, p.per, kRing<2, 2>);
  return UNIT_OK;
}
