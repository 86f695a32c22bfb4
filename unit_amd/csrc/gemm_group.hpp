// GEMM for problems that do not fill the chip with large tiles: one small output tile per workgroup, KG groups of
// WX x WY waves each on its own share of the reduction, operands global -> LDS by direct loads into a ring per group.
//
// What bounds such a problem is latency and the 57-59 B/clk a CU takes from its L2, not the matrix cores: few tiles
// mean few CUs with work, so the reduction is shared inside the workgroup (KG rings of loads in flight on one tile, partial
// tiles summed in LDS in group order: deterministic, no zero fill, no atomics) before it is split across workgroups.
//
// Any reduction length that keeps rows 16-byte aligned: all loads are raw buffer loads, and a lane whose chunk lies past
// the end of its row is sent out of range, where the load stores zeros.
//
// Y operand (YM):
//   Y_ROWS    (N, K) rows, K-contiguous: row-major int8 weights, the fp16 b re-laid by unit_gemm_f16_prepare_b;
//   Y_COLS    (K, N) fp16 as the reference's GEMM gives b: its tile lands as it lies, [k][columns], and fragments come
//             out of it with the LDS transposing read.  N a multiple of 4: the last chunk of a row whose N is 4 mod 8
//             is fetched 4 columns early (it stays inside the row) and its reader looks 8 bytes further;
//   Y_VNNI    (N/128, K/4, 128, 4) int8 pre-pack: lands as [k / 4][row][4 bytes], a fragment is four dwords 4 * BY
//             bytes apart.  Past the end of the reduction it holds the next block's weights: the activations there are
//             zeros, and what a shifted zero (-128) times such a weight adds, its weight sum takes away.
#pragma once
#include "host.hpp"
#include "mma_dma.hpp"

namespace unit {

enum { Y_ROWS = 0, Y_COLS = 1, Y_VNNI = 2 };
enum { C_STORE = 0, C_ATOMIC = 1, C_PLANES = 2 };  // several k-splits: added into a zeroed c, or one fp32 plane each

struct GroupGemm {
  const char *x, *y;
  u32 xbytes, ybytes;  // operand sizes (bounds of the buffer loads)
  int M, N;
  int kb;    // reduction bytes per row of x
  int ldy;   // Y_ROWS: bytes per row; Y_COLS: bytes per k row
  const int *ysum;  // WS_Y_GIVEN
  void *c;
  int mode;
  size_t plane;  // C_PLANES: bytes per plane
};

template <int TX_, int TY_, int WX_, int WY_, int KG_, int BKB_, int NST_>
struct GroupTile {
  static constexpr int TX = TX_, TY = TY_, WX = WX_, WY = WY_, KG = KG_, BKB = BKB_, NST = NST_;
  static constexpr int BX = 32 * TX * WX, BY = 32 * TY * WY;
  static constexpr int NWG = WX * WY, NW = NWG * KG, NT = 64 * NW;
  static constexpr int CPR = BKB / 16, KK = BKB / 32, RPL = 64 / CPR;  // chunks per row, k-steps per stage, rows per load
  static constexpr int XL = BX / RPL / NWG, YL = BY / RPL / NWG, LPS = XL + YL;  // direct loads per wave and stage
  static constexpr int XBYTES = BX * BKB, STAGE = (BX + BY) * BKB, RING = NST * STAGE;
  static constexpr int PITCH = BY + 4;            // elements per row of a parked partial tile
  static constexpr int PARK = BX * PITCH * 4;     // bytes per group
  static constexpr int BACK = KG * (PARK + WX * BY * 4);  // parked tiles, then weight sums
  static constexpr int LDS = KG * RING > BACK ? KG * RING : BACK;
  static_assert(BX % (RPL * NWG) == 0 && BY % (RPL * NWG) == 0, "direct loads split evenly over the waves of a group");
  static_assert(KK % 2 == 0 && NST >= 3 && NST <= 6 && NT <= 1024 && NT >= BY && LDS <= kMaxLds && (BY & (BY - 1)) == 0 && (WX & (WX - 1)) == 0 && BY <= 128, "group tile");
};

template <class Op, class T, int YM, int WS, bool OUT_F16>
__global__ __launch_bounds__(T::NT) void gemm_group(GroupGemm p, GridMap gm) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int TX = T::TX, TY = T::TY, NST = T::NST, KK = T::KK, XL = T::XL, YL = T::YL, BKB = T::BKB, BY = T::BY;
  constexpr bool kInt = Op::kInt;
  static_assert(kInt == (WS != WS_NONE) && (YM != Y_COLS || !kInt) && (YM != Y_VNNI || WS == WS_Y), "operand forms");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int grp = wave / T::NWG, wg = wave % T::NWG;
  const int wx = wg % T::WX, wy = wg / T::WX;
  const int l32 = lane & 31, half = lane >> 5;

  int bx, by, split;
  gm.locate(blockIdx.x, bx, by, split);
  const int x0 = bx * T::BX, y0 = by * BY;
  // stages [b0, b1) of this k-split, [s0, s0 + n) of this group
  const int nk = (p.kb + BKB - 1) / BKB;
  const int b0 = (int)((long)nk * split / gm.splits), b1 = (int)((long)nk * (split + 1) / gm.splits);
  const int s0 = b0 + (b1 - b0) * grp / T::KG, n = b0 + (b1 - b0) * (grp + 1) / T::KG - s0;
  const int rounds = (b1 - b0 + T::KG - 1) / T::KG;

  auto raw_buffer = [](const char *ptr, u32 bytes) {
    const unsigned long long base = (unsigned long long)ptr;
    v4i r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(u32)base);
    r[1] = __builtin_amdgcn_readfirstlane((int)((u32)(base >> 32) & 0xffffu));
    r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
    r[3] = 0x00020000;
    return r;
  };
  const v4i xsrc = raw_buffer(p.x, p.xbytes), ysrc = raw_buffer(p.y, p.ybytes);
  char *ring = lds + grp * T::RING;
  const u32 ring_addr = (u32)(uintptr_t)(lptr_t)ring;
  constexpr u32 kOutside = 0x80000000u;  // operands stay below 2^31 bytes

  // lane offsets of this wave's loads of a stage; *_last: of the reduction's last stage, whose chunks may lie past its end
  u32 xoff[XL], xlast[XL], yoff[YL], ylast[YL];
  const int tail0 = (nk - 1) * BKB;
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = (wg * XL + i) * T::RPL + lane / T::CPR, c = ((lane % T::CPR) ^ swz<BKB>(row)) << 4;
    xoff[i] = (u32)min(x0 + row, p.M - 1) * (u32)p.kb + (u32)c;
    xlast[i] = tail0 + c < p.kb ? xoff[i] : kOutside;
  }
  // Y_COLS: XOR of the 16-byte chunk position inside a k row, so that the four k rows of a transposing read fall into
  // different bank groups (rows of 64, 128 or 256 bytes)
  auto colswz = [](int krow) { return BY >= 128 ? 4 * (krow & 3) : BY == 64 ? 4 * ((krow >> 1) & 1) : 0; };
  constexpr int CPY = YM == Y_COLS ? BY / 8 : BY / 4;  // Y_COLS, Y_VNNI: 16-byte chunks per row of the tile
  u32 ysoff0 = 0, ystep = BKB;  // scalar offset of stage 0, and from stage to stage
  if constexpr (YM == Y_COLS) ystep = (u32)(BKB / 2) * (u32)p.ldy;
  if constexpr (YM == Y_VNNI) {
    ystep = BKB / 4 * 512;
    ysoff0 = (u32)(y0 >> 7) * (u32)(p.kb >> 2) * 512u + (u32)(y0 & 127) * 4u;
  }
#pragma unroll
  for (int i = 0; i < YL; ++i) {
    if constexpr (YM == Y_ROWS) {
      const int row = (wg * YL + i) * T::RPL + lane / T::CPR, c = ((lane % T::CPR) ^ swz<BKB>(row)) << 4;
      yoff[i] = (u32)min(y0 + row, p.N - 1) * (u32)p.ldy + (u32)c;
      ylast[i] = tail0 + c < p.kb ? yoff[i] : kOutside;
    } else {
      const int row = (wg * YL + i) * (64 / CPY) + lane / CPY;
      if constexpr (YM == Y_COLS)
        yoff[i] = (u32)row * (u32)p.ldy + (u32)min((y0 / 8 + ((lane % CPY) ^ colswz(row))) * 16, 2 * p.N - 16);
      else
        yoff[i] = (u32)row * 512u + (u32)(lane % CPY) * 16u;
      ylast[i] = yoff[i];  // k rows past the end lie past the operand, or are harmless (above)
    }
  }
  auto issue = [&](int it, int slot) __attribute__((always_inline)) {  // the loads of this group's stage `it`, slot = it % NST
    const int st = s0 + it;
    const bool last = st == nk - 1;
    const u32 buf = ring_addr + (u32)slot * T::STAGE;
#pragma unroll
    for (int i = 0; i < XL; ++i)
      dma_buffer_16(buf + (wg * XL + i) * 1024, last ? xlast[i] : xoff[i], xsrc, (u32)st * BKB);
#pragma unroll
    for (int i = 0; i < YL; ++i)
      dma_buffer_16(buf + T::XBYTES + (wg * YL + i) * 1024, last ? ylast[i] : yoff[i], ysrc, ysoff0 + (u32)st * ystep);
  };
#pragma unroll
  for (int s = 0; s < NST; ++s)
    if (s < n) issue(s, s);

  // given weight sums: fetched here, so that the latency hides behind the loop (one k-split adds the whole sum)
  int given = 0;
  if constexpr (WS == WS_Y_GIVEN) {
    const int t = threadIdx.x;
    if (t < BY && y0 + t < p.N && split == 0) given = p.ysum[y0 + t];
  }

  typename Op::acc_t acc[TX][TY];
#pragma unroll
  for (int i = 0; i < TX; ++i)
#pragma unroll
    for (int j = 0; j < TY; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  int wsy[TY];
#pragma unroll
  for (int j = 0; j < TY; ++j) wsy[j] = 0;

  const int xrow = wx * (TX * 32) + l32, yrow = wy * (TY * 32) + l32;
  const int xsw = swz<BKB>(xrow), ysw = swz<BKB>(yrow);
  int ytr[TY];  // Y_COLS: what this lane hands to the transposing reads of fragment j, k-step 0
  if constexpr (YM == Y_COLS) {
    const int jrow = (lane & 15) >> 2, q = lane & 3, g16 = (lane >> 4) & 1;
#pragma unroll
    for (int j = 0; j < TY; ++j) {
      const int c = wy * (TY * 4) + j * 4 + 2 * g16 + (q >> 1);
      const int col4 = (y0 >> 2) + 2 * c + (q & 1);  // this lane's four columns, in units of four
      const int early = (p.N & 4) && col4 == (p.N >> 2) - 1 ? 8 : 0;  // they lie in a chunk that was fetched 4 columns early
      ytr[j] = (8 * half + jrow) * (BY * 2) + ((c ^ colswz(jrow)) << 4) + (q & 1) * 8 + early;
    }
  }
  auto load_y = [&](const char *tile, int kk, int j) -> v4i {
    if constexpr (YM == Y_ROWS) {
      return *reinterpret_cast<const v4i *>(tile + (yrow + j * 32) * BKB + (((2 * kk + half) ^ ysw) << 4));
    } else if constexpr (YM == Y_COLS) {
      typedef __attribute__((address_space(3))) v4s *trptr_t;
      typedef short v8s __attribute__((ext_vector_type(8)));
      const char *src = tile + ytr[j] + kk * 16 * (BY * 2);
      const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(src));
      const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(src + 4 * (BY * 2)));
      return __builtin_bit_cast(v4i, (v8s)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const int *src = reinterpret_cast<const int *>(tile + ((8 * kk + 4 * half) * BY + yrow + j * 32) * 4);
      return v4i{src[0], src[BY], src[2 * BY], src[3 * BY]};
    }
  };

  v4i xf[2][TX], yf[2][TY];
  auto load_frags = [&](int slot, int kk, int f) __attribute__((always_inline)) {
    const char *xt = ring + slot * T::STAGE, *yt = xt + T::XBYTES;
#pragma unroll
    for (int i = 0; i < TX; ++i)
      xf[f][i] = *reinterpret_cast<const v4i *>(xt + (xrow + i * 32) * BKB + (((2 * kk + half) ^ xsw) << 4));
#pragma unroll
    for (int j = 0; j < TY; ++j) yf[f][j] = load_y(yt, kk, j);
  };
  auto mma_step = [&](int f, int turn) __attribute__((always_inline)) {
    if constexpr (kInt) {
#pragma unroll
      for (int i = 0; i < TX; ++i) xf[f][i] ^= (int)0x80808080;
    }
    if constexpr (WS == WS_Y) {
      // the WX waves that read the same Y fragments take turns to sum them (1024 x 4096 x 4096: 31.7 us when each did)
      if ((turn & (T::WX - 1)) == wx) {
#pragma unroll
        for (int j = 0; j < TY; ++j)
#pragma unroll
          for (int d = 0; d < 4; ++d) wsy[j] = __builtin_amdgcn_sdot4(yf[f][j][d], 0x01010101, wsy[j], false);
      }
    }
#pragma unroll
    for (int i = 0; i < TX; ++i)
#pragma unroll
      for (int j = 0; j < TY; ++j) acc[i][j] = Op::mma(xf[f][i], yf[f][j], acc[i][j]);
  };
  // wait until only the `behind` youngest stages' loads are in flight
  auto wait_stages = [&](int behind) __attribute__((always_inline)) {
    if (NST > 5 && behind == 4) {
      UNIT_WAIT_VMCNT(4 * T::LPS);
    } else if (NST > 4 && behind == 3) {
      UNIT_WAIT_VMCNT(3 * T::LPS);
    } else if (NST > 3 && behind == 2) {
      UNIT_WAIT_VMCNT(2 * T::LPS);
    } else if (behind == 1) {
      UNIT_WAIT_VMCNT(T::LPS);
    } else {
      UNIT_WAIT_VMCNT(0);
    }
  };
  // Fragments are read one k-step ahead of the MFMAs, across the stage boundary: before a stage's last k-step the next
  // stage has landed, everybody has read this one, and its buffer takes stage it + NST.
  auto boundary = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads are done
    if constexpr (T::NWG > 1) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (n >= NST) {
    UNIT_WAIT_VMCNT((NST - 1) * T::LPS);
  } else {
    wait_stages(n - 1);
  }
  if constexpr (T::NWG > 1) __builtin_amdgcn_s_barrier();
  if (n > 0) load_frags(0, 0, 0);
  int it = 0, slot = 0;
  for (; it + NST < n; ++it) {  // steady state
    const int next = slot + 1 == NST ? 0 : slot + 1;
#pragma unroll
    for (int kk = 0; kk + 1 < KK; ++kk) {
      load_frags(slot, kk + 1, (kk + 1) & 1);
      mma_step(kk & 1, it * KK + kk);
    }
    UNIT_WAIT_VMCNT((NST - 2) * T::LPS);
    boundary();
    issue(it + NST, slot);
    load_frags(next, 0, 0);
    mma_step((KK - 1) & 1, it * KK + KK - 1);
    slot = next;
  }
  for (; it < rounds; ++it) {  // nothing left to fetch; groups with fewer stages keep the others company at the barriers
    const int next = slot + 1 == NST ? 0 : slot + 1;
    if (it < n) {
#pragma unroll
      for (int kk = 0; kk + 1 < KK; ++kk) {
        load_frags(slot, kk + 1, (kk + 1) & 1);
        mma_step(kk & 1, it * KK + kk);
      }
    }
    if (it + 1 < n) wait_stages(n - 2 - it);
    boundary();
    if (it < n) {
      if (it + 1 < n) load_frags(next, 0, 0);
      mma_step((KK - 1) & 1, it * KK + KK - 1);
    }
    slot = next;
  }

  // ---- the groups' partial tiles meet in LDS, row-major, and all waves write the sums 16 bytes per lane
  __syncthreads();
  using elem_t = typename Op::out_t;
  using elem4_t = typename Op::out4_t;
  {
    elem_t *mine = reinterpret_cast<elem_t *>(lds + grp * T::PARK);
#pragma unroll
    for (int i = 0; i < TX; ++i)
#pragma unroll
      for (int j = 0; j < TY; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          mine[(wx * (TX * 32) + i * 32 + 8 * (r >> 2) + 4 * half + (r & 3)) * T::PITCH + yrow + j * 32] = acc[i][j][r];
    if constexpr (WS == WS_Y) {
      int *sums = reinterpret_cast<int *>(lds + T::KG * T::PARK) + (grp * T::WX + wx) * BY;
#pragma unroll
      for (int j = 0; j < TY; ++j) {
        const int both = wsy[j] + __shfl_xor(wsy[j], 32);
        if (half == 0) sums[yrow + j * 32] = both;
      }
    }
    if constexpr (WS == WS_Y_GIVEN) {
      if (threadIdx.x < BY) reinterpret_cast<int *>(lds + T::KG * T::PARK)[threadIdx.x] = given;
    }
  }
  __syncthreads();
  const int *sums = reinterpret_cast<const int *>(lds + T::KG * T::PARK);
  char *const c = static_cast<char *>(p.c) + (p.mode == C_PLANES ? (size_t)split * p.plane : 0);
  const __amdgpu_buffer_rsrc_t cbuf = result_buffer(c);
  if (p.mode == C_ATOMIC) {
    // one element per lane: an instruction adds to consecutive elements of a row, whole lines at the memory side, where
    // four elements per lane took four instructions to every line (128 x 768 x 8192 fp16 in nine splits 19.8 -> 11.2 us)
    for (int u = threadIdx.x; u < T::BX * BY; u += T::NT) {
      const int row = u / BY, col = u % BY;
      const int m = x0 + row, col_n = y0 + col;
      if (m >= p.M || col_n >= p.N) continue;
      elem_t v = *reinterpret_cast<const elem_t *>(lds + (row * T::PITCH + col) * 4);
#pragma unroll
      for (int g = 1; g < T::KG; ++g) v += *reinterpret_cast<const elem_t *>(lds + g * T::PARK + (row * T::PITCH + col) * 4);
      const u32 idx = (u32)m * (u32)p.N + (u32)col_n;
      if constexpr (kInt) {
        int w = sums[col];
#pragma unroll
        for (int g = 1; g < (WS == WS_Y ? T::KG * T::WX : 1); ++g) w += sums[g * BY + col];
        atomicAdd(reinterpret_cast<int *>(c) + idx, v + (w << 7));
      } else {
        unsafeAtomicAdd(reinterpret_cast<float *>(c) + idx, v);
      }
    }
    return;
  }
  constexpr int Q = BY / 4;  // quads per row
  for (int u = threadIdx.x; u < T::BX * Q; u += T::NT) {
    const int row = u / Q, col = (u % Q) * 4;
    const int m = x0 + row, col_n = y0 + col;
    if (m >= p.M || col_n >= p.N) continue;
    elem4_t v = *reinterpret_cast<const elem4_t *>(lds + (row * T::PITCH + col) * 4);
#pragma unroll
    for (int g = 1; g < T::KG; ++g) v += *reinterpret_cast<const elem4_t *>(lds + g * T::PARK + (row * T::PITCH + col) * 4);
    if constexpr (WS != WS_NONE) {
      v4i w = *reinterpret_cast<const v4i *>(sums + col);
#pragma unroll
      for (int g = 1; g < (WS == WS_Y ? T::KG * T::WX : 1); ++g) w += *reinterpret_cast<const v4i *>(sums + g * BY + col);
      v += w << 7;
    }
    const u32 idx = (u32)m * (u32)p.N + (u32)col_n;
    if (OUT_F16 && p.mode == C_STORE) {
      typedef _Float16 v4h __attribute__((ext_vector_type(4)));
      const v4h h = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, h), cbuf, (int)(idx * 2u), 0, kRowPolicy);
    } else {
      store_result<kRowPolicy>(cbuf, idx * 4u, v);
    }
  }
}

// splits > 1 with C_ATOMIC zero-fills c first (M * N * 4 a multiple of 16); with C_PLANES c is the workspace.
template <class Op, class T, int YM, int WS, bool OUT_F16>
int run_gemm_group(const char *what, const char *tag, GroupGemm p, int splits, hipStream_t s) {
  auto kern = gemm_group<Op, T, YM, WS, OUT_F16>;
  static thread_local bool allowed = false;  // the opt-in for > 64 KiB of dynamic LDS is sticky per kernel
  if (!allowed && T::LDS > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    allowed = true;
  }
  const int nk = ceil_div(p.kb, T::BKB), gx = ceil_div(p.M, T::BX), gy = ceil_div(p.N, T::BY);
  splits = splits < 1 ? 1 : (splits > nk ? nk : splits);
  if (splits == 1) {
    if (p.mode == C_ATOMIC) p.mode = C_STORE;
  } else if (p.mode == C_ATOMIC) {
    const size_t n16 = (size_t)p.M * p.N * 4 / 16;
    hipLaunchKernelGGL(zero_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, static_cast<v4i *>(p.c), n16);
  }
  const GridMap gm = GridMap::make(gx, gy, gx < 4 ? gx : 4, splits);
  set_variant("%s_x%d_y%d_k%d_w%dx%d_g%d_r%d%s_s%d", tag, T::BX, T::BY, T::BKB, T::WX, T::WY, T::KG, T::NST,
              OUT_F16 ? "_h" : "", splits);
  hipLaunchKernelGGL(kern, dim3(gm.total), dim3(T::NT), T::LDS, s, p, gm);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK : fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
}

// ---- which tile, and how many k-splits
//
// Estimated time (us) of a launch of `tiles` output tiles in `splits` k-ranges: the busiest of the 256 CUs runs
// w = ceil(tiles * splits / 256) workgroups, per_cu of them at a time (LDS), each t_tile plus t_stage per stage of its
// reduction share -- or, side by side, share per stage and workgroup (operand delivery into the CU).  Not below the
// padded work at `rate` (kilobyte-products per us: with most CUs busy the clock gives).  Where the operand + result
// traffic at `hbm` TB/s is the longer of the two, a third of the difference hides behind it (4405 x 1536 x 64 fp16: 64 x 128
// tiles, 60 of them in a second round, 7.1 us, 128 x 128 in one 5.7).  The constants are least-squares fits to 4200 timings (70 fp16 and 60 int8 shapes per weight
// layout, 1 x 836 x 2736 to 8192 x 8192 x 2048, every tile and up to 16 splits): the pick is on average 3 % above the
// best measured tile.  Against the 128 x 128 tiles with k-splits by atomics and the register pipelines that served these
// shapes, us a call in a row of them: fp16 1000 x 1516 x 1096 24.8 -> 10.3, 64 x 4096 x 4096 15.6 -> 14.0 (b prepared
// 15.9 -> 11.5), int8 packed 128 x 768 x 3072 12.4 -> 6.4, 1 x 4096 x 4096 15.9 -> 6.8, 1467 x 1152 x 976 16.2 -> 9.3;
// geometric mean over random shapes 1.5 x.
struct GroupCost {
  int bx, by, kg, per_cu;
  float launch, tile, stage, share, hbm, rate;
};
constexpr GroupCost kGroupCosts[] = {
    {32, 32, 8, 1, 1.0f, 1.65f, 0.587f, 0.587f, 4.7f, 1e6f},   // 0: eight groups of one wave
    {32, 32, 4, 2, 1.8f, 1.00f, 0.223f, 0.280f, 4.9f, 224.f},  // 1: four groups of one wave, two workgroups per CU
    {32, 64, 4, 1, 1.0f, 2.03f, 0.374f, 0.374f, 4.6f, 1e6f},   // 2: four groups of two waves
    {64, 64, 2, 2, 1.0f, 2.40f, 0.212f, 0.239f, 5.0f, 467.f},  // 3: two groups of four waves
    {64, 128, 1, 3, 1.0f, 2.70f, 0.169f, 0.201f, 4.8f, 593.f}, // 4: four waves
    {128, 128, 1, 2, 1.0f, 3.17f, 0.247f, 0.254f, 4.2f, 662.f},  // 5: eight waves (Y_VNNI: four)
    {256, 128, 1, 1, 3.6f, 3.36f, 0.482f, 0.482f, 3.6f, 811.f},  // 6: eight waves
};
constexpr int kGroupTiles = sizeof(kGroupCosts) / sizeof(kGroupCosts[0]);

struct GroupPlan {
  int tile, splits;
  float us;
};

inline float group_cost(const GroupCost &g, long M, long N, long kb, int splits, long operand_bytes, long out_bytes) {
  const long tiles = (M + g.bx - 1) / g.bx * ((N + g.by - 1) / g.by);
  const long nk = (kb + 63) / 64, share = (nk + splits - 1) / splits, n = (share + g.kg - 1) / g.kg;
  const long w = (tiles * splits + 255) / 256, full = w / g.per_cu, rest = w % g.per_cu;
  auto side_by_side = [&](long k) { return g.tile + n * (g.stage > k * g.share ? g.stage : k * g.share); };
  float t = g.launch + full * side_by_side(g.per_cu) + (rest ? side_by_side(rest) : 0.f);
  const float work = g.launch + g.tile + (float)tiles * g.bx * g.by * kb / (g.rate * 1e6f);
  const float mem = 2.f + (operand_bytes + (float)out_bytes * splits) / (g.hbm * 1e6f);
  t = t > work ? t : work;
  return ((t > mem ? t : mem) + 0.5f * t) / 1.5f;
}

inline long tiles_of_128(int M, int N) { return (long)ceil_div(M, 128) * ceil_div(N, 128); }

// extra + out_bytes * splits / rate: what a split launch costs besides (zero fill and atomics, or the pass that adds
// the planes).  At least min_splits ranges, where an operator shares its reduction between workgroups in any case.
struct SplitCost {
  float extra, rate;
};
constexpr SplitCost kAtomicSplits{2.4f, 1.2f}, kPlaneSplits{2.8f, 4.5f};

inline GroupPlan plan_group(int M, int N, int kb, int min_splits, int max_splits, SplitCost split, int out_elem = 4) {
  GroupPlan best{0, 1, 1e30f};
  const long nk = ceil_div(kb, 64), operands = (long)M * kb + (long)N * kb, out = (long)M * N * out_elem;
  if (min_splits > nk) min_splits = (int)nk;
  if (max_splits < min_splits) max_splits = min_splits;
  for (int i = 0; i < kGroupTiles; ++i) {
    const GroupCost &g = kGroupCosts[i];
    const long tiles = (long)ceil_div(M, g.bx) * ceil_div(N, g.by);
    for (int s = min_splits; s <= max_splits && s <= nk; s = s < 4 ? s + 1 : s * 3 / 2) {  // 1 2 3 4 6 9 13 19
      if (s > min_splits && (tiles * s > 768 || nk / s < 6)) break;
      const float us = group_cost(g, M, N, kb, s, operands, out) + (s > 1 ? split.extra + out * (float)s / (split.rate * 1e6f) : 0.f);
      if (us < best.us) best = GroupPlan{i, s, us};
    }
  }
  return best;
}

// Products of more than one 128 x 128 tile per CU and at most one of 256 x 128: the large tile with 128-byte stages.  The
// estimate sees two of the small tiles side by side on some CUs at nearly the cost of one; they take in half as much again
// per result, and in 64-byte stages at that (two rings of 128 bytes do not fit a CU).  us of 128 x 128 / 256 x 128 in 64- / in 128-byte
// stages: fp16 2304 x 2048 x 2056 42.5 / 39.1 / 32.8, prepared 53.8 / 43.8 / 34.7, 2600 x 1900 x 3000 64.0 / 58.3 / 47.1, 5472 x 1096 x
// 712 prepared 23.2 / 21.9 / 19.8; int8 2304 x 2048 x 2064 31.3 / 26.9 / 24.2, 829 x 5848 x 2576 37.7 / 32.0 / 28.0, 711 x 5480 x 1024 15.7 /
// 15.1 / 14.8.  The other way from 640 bytes of reduction down (4317 x 1536 x 320 fp16 12.5 / - / 12.9), on packed weights
// (5400 x 1408 x 1072 19.1 / 20.8 / 21.7) and where 64 x 128 tiles are the estimate's choice, up to 2 KiB (1566 x 2548 x 672 14.8 / - /
// 16.9).  Left where they were: 301 - 306
// small tiles of a result whose last row of large ones is cut off, from 2 KiB on, for which tests name the small ones (2180 x 2052 x 2056
// fp16 43.2 us, 33.0 on the large ones; int8 2180 x 2176 x 2064 31.4 and 24.1).
inline bool one_wide_tile_per_cu(int M, int N, int kb) {
  const long half = tiles_of_128(M, N), tiles = (long)ceil_div(M, 256) * ceil_div(N, 128);
  return half > 256 && tiles <= 256 && kb >= 768 && !(half > 300 && tiles <= 153 && M % 256 && kb >= 2048);
}
inline GroupPlan prefer_wide_tile(const GroupPlan &plan, int M, int N, int kb) {
  return plan.splits == 1 && (plan.tile == 5 || (plan.tile == 4 && kb >= 2048)) && one_wide_tile_per_cu(M, N, kb) ? GroupPlan{6, 1, plan.us} : plan;
}

// The same estimate for 256 x 256 tiles of eight waves: per round of 256 tiles 3 us plus 24.9 us per 2 KiB of
// reduction (18.7 with at most 200 CUs busy), and the result at 6.4 TB/s.
inline float large_tile_cost(int M, int N, int kb) {
  const long tiles = (long)ceil_div(M, 256) * ceil_div(N, 256);
  return 2.f + (float)((tiles + 255) / 256) * (3.f + (tiles <= 200 ? 18.7f : 24.9f) * kb / 2048) + (float)M * N * 4 / 6.4e6f;
}

// Stages of 128 bytes instead of 64 while there is at most one tile per CU.  A row of a stage is then a whole cache line
// (with 64 bytes every line is asked for twice, half of it each time), and the waves meet at half as many barriers.  Their
// rings leave room for one workgroup per CU (96 - 144 KiB), where those of 64-byte stages have up to three: past 256 tiles
// that is worth more.  us on operands that change from call to call, 64 / 128 bytes: fp16 700 x 2304 x 3008 20.5 / 16.9,
// 900 x 1664 x 1600 12.6 / 10.8, prepared 500 x 2048 x 2048 11.3 / 9.3, 1500 x 1536 x 1504 17.4 / 15.1; int8 packed 900 x
// 1664 x 1600 11.4 / 9.9, 1500 x 1536 x 1504 14.7 / 11.8, row-major 700 x 2304 x 3008 16.0 / 13.3; geometric mean over the 84 of
// 231 random products that it takes 1.11, lowest 0.98.
// The other way: 512 tiles of 64 x 64 (2000 x 1024 x 512) 6.8 / 7.9, 640 bytes of reduction (702 x 1216 x 320) 4.3 / 4.5 and, on
// 32 x 32 tiles, 1088 (93 x 2112 x 544) 3.75 / 3.88, b by columns on 32 x 32 tiles, whose rows of b stay 64 bytes, 15 x 2560 x 5488
// 17.6 / 20.1.  b by columns whose rows end inside lines, on 64 x 128 tiles, up to 3 KiB of reduction: 1000 x 1516 x 1096 10.34 /
// 10.41 (fp32 result 10.7 / 11.0), 966 x 1804 x 856 9.6 / 10.0, 822 x 2280 x 1016 10.4 / 10.7, others down to 0.93; from 3 KiB on
// 0.91 - 1.01.  int8 products of up to 64 rows and 4096 columns, where a launch's latency is most of it, up to 3 KiB:
// 64 x 4096 x 1536 prepared 5.0 / 5.4, 1 x 4096 x 2048 4.8 / 5.2, packed 23 x 2944 x 2240 5.0 / 5.3; from there on 64 x 4096 x 4096
// row-major 7.8 / 6.3, packed 7.1 / 6.5, 1 x 4096 x 4096 6.2 / 6.0, 57 x 3712 x 8112 prepared 15.9 / 12.6 (64 x 8192 x 1536 6.0 / 4.9).
template <class Op, int YM>
bool group_wide_stages(const GroupGemm &p, const GroupPlan &plan) {
  const GroupCost &g = kGroupCosts[plan.tile];
  const int least = plan.tile == 6 ? 768 : plan.tile >= 2 ? 960 : Op::kInt && p.M <= 64 && p.N <= 4096 ? 3072 : 1536;
  return plan.splits == 1 && p.kb >= least && (long)ceil_div(p.M, g.bx) * ceil_div(p.N, g.by) <= 256 &&
         !(YM == Y_COLS && (plan.tile < 2 || (plan.tile == 4 && p.kb < 3072 && p.ldy % 128)));
}

template <class Op, int YM, int WS, bool OUT_F16>
int run_group_plan(const char *what, const char *tag, const GroupGemm &p, const GroupPlan &plan, hipStream_t s) {
  using Wide = std::conditional_t<YM == Y_VNNI, GroupTile<2, 2, 2, 2, 1, 64, 4>, GroupTile<1, 2, 4, 2, 1, 64, 4>>;
  if (group_wide_stages<Op, YM>(p, plan)) {
    switch (plan.tile) {
      case 0:
      case 1:
        if constexpr (YM != Y_COLS) return run_gemm_group<Op, GroupTile<1, 1, 1, 1, 4, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
        break;
      case 2: return run_gemm_group<Op, GroupTile<1, 1, 1, 2, 4, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
      case 3: return run_gemm_group<Op, GroupTile<1, 1, 2, 2, 2, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
      case 4: return run_gemm_group<Op, GroupTile<1, 2, 2, 2, 2, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
      case 5: return run_gemm_group<Op, GroupTile<1, 2, 4, 2, 1, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
      case 6:
        if constexpr (YM != Y_VNNI) return run_gemm_group<Op, GroupTile<2, 2, 4, 2, 1, 128, 3>, YM, WS, OUT_F16>(what, tag, p, 1, s);
        break;
      default: break;
    }
  }
  switch (plan.tile) {
    case 0: return run_gemm_group<Op, GroupTile<1, 1, 1, 1, 8, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    case 1: return run_gemm_group<Op, GroupTile<1, 1, 1, 1, 4, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    case 2: return run_gemm_group<Op, GroupTile<1, 1, 1, 2, 4, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    case 3: return run_gemm_group<Op, GroupTile<1, 1, 2, 2, 2, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    case 4: return run_gemm_group<Op, GroupTile<1, 2, 2, 2, 1, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    case 5: return run_gemm_group<Op, Wide, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
    default: return run_gemm_group<Op, GroupTile<2, 2, 4, 2, 1, 64, 4>, YM, WS, OUT_F16>(what, tag, p, plan.splits, s);
  }
}

}  // namespace unit
