// The first convolution of an image network, planar in and out: x (N, C, H, W) s8 with C <= 4, weights in prepared form
// (4-channel blocks), out (N, out_channels, OH, OW) = (conv(x, w) + bias) * scale.  The printed graph runs it as
// layout_transform, convolution, layout_transform (apps/cpu/relay/result.log:6803-6838); here it is one launch.
//
// What bounds it is the result (51 MB at 16 x 3 x 224 x 224, 64 channels, 7 x 7, stride 2: 8 us at the rate of a fill),
// so everything in front of the stores has to be short.  A workgroup takes 32 TY x 4 consecutive output pixels of one
// image and all or a third / half of the channels: it lays the input rows under its window out in LDS, once, as 4-byte pixels with the
// zero padding in place, beside the weight fragments.  A k-step (one window row) is then one 16-byte LDS read per
// 32 pixels -- the direct kernel on a packed copy spends four masked 4-byte gathers from memory there, and a
// launch and a round trip through memory on the copy.
#include "conv_plan.hpp"
#include "conv_prepare.hpp"
#include "mma_dma.hpp"

namespace unit {
namespace {

struct PlanarC4 {
  const char *x, *w;
  const int *bias;
  void *out;
  int scale;
  int C, H, W, OW, OHW, KH, sh, sw, dh, pt, pl, oc;
  int quads;  // 16-byte groups of four pixels per patch row
  FastDiv by_quads, by_ow, by_tiles, by_kg;
};

typedef u32 word_at_t __attribute__((aligned(1)));

// NC: input channels read (3, or 4 with those past C masked)
template <int TX, int TY, int NC>
__global__ __launch_bounds__(256) void conv_planar_c4_kernel(PlanarC4 p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int PT = 128 * TY;
  const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int rest, kg, n, tile, oh0, oh1, rem;
  p.by_kg.divmod((int)blockIdx.x, rest, kg);
  p.by_tiles.divmod(rest, n, tile);
  const int p0 = tile * PT, last = min(p0 + PT, p.OHW) - 1;
  p.by_ow.divmod(p0, oh0, rem);
  p.by_ow.divmod(last, oh1, rem);
  const int wbytes = TX * p.KH * 1024, pitch = p.quads * 16;
  int *bias = reinterpret_cast<int *>(lds + wbytes);
  char *patch = lds + wbytes + TX * 128;

  // the weight fragments of the workgroup's TX blocks are consecutive in the prepared buffer
  const char *wsrc = p.w + (size_t)kg * wbytes;
  for (int s = wave; s < TX * p.KH; s += 4)
    __builtin_amdgcn_global_load_lds((gptr_t)(wsrc + s * 1024 + lane * 16), (lptr_t)(lds + s * 1024), 16, 0, 0);
  if (threadIdx.x < TX * 32) {
    const int c = kg * (TX * 32) + (int)threadIdx.x;
    bias[threadIdx.x] = p.bias != nullptr && c < p.oc ? p.bias[c] : 0;
  }

  // patch: rows ih0 .. of the image, column 0 = image column -pl; four groups of four pixels in flight per thread.  A
  // group's word starts at the nearest place inside the row and is shifted; rows outside the image read row 0, masked.
  const int ih0 = oh0 * p.sh - p.pt, groups = ((oh1 - oh0) * p.sh + (p.KH - 1) * p.dh + 1) * p.quads;
  const size_t plane = (size_t)p.H * p.W;
  const char *img = p.x + (size_t)n * p.C * plane;
  for (int u0 = threadIdx.x; u0 < groups; u0 += 1024) {
    u32 v[4][4];
    int shift[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int r, q;
      p.by_quads.divmod(min(u0 + 256 * k, groups - 1), r, q);
      const int ih = ih0 + r, iw = 4 * q - p.pl;
      const int at = min(max(iw, 0), p.W - 4);
      const bool in = (u32)ih < (u32)p.H && iw > -4 && iw < p.W;
      shift[k] = in ? iw - at : 4;
      const char *src = img + ((size_t)(in ? ih : 0) * p.W + at);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[k][c] = c < NC ? *reinterpret_cast<const word_at_t *>(src + (c < p.C ? c : 0) * plane) : 0u;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int u = u0 + 256 * k;
      // bytes of the word that lie outside the row fall out: left of it (shift < 0) or right of it
      const u32 up = shift[k] < 0 ? (u32)(-8 * shift[k]) : 0u, down = shift[k] > 0 ? (u32)(8 * shift[k]) : 0u;
      u32 w[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        w[c] = down < 32 ? (v[k][c] >> (down & 31)) << up : 0u;
        if (c >= p.C) w[c] = 0u;
      }
      const u32 a0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), a1 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
      const u32 b0 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), b1 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
      if (u < groups)
        *reinterpret_cast<v4u *>(patch + u * 16) =
            v4u{__builtin_amdgcn_perm(b0, a0, 0x05040100u), __builtin_amdgcn_perm(b0, a0, 0x07060302u),
                __builtin_amdgcn_perm(b1, a1, 0x05040100u), __builtin_amdgcn_perm(b1, a1, 0x07060302u)};
    }
  }

  int yoff[TY];  // of this lane's pixel: its window's first row, taps 4 half .. + 3
#pragma unroll
  for (int j = 0; j < TY; ++j) {
    int oh, ow;
    p.by_ow.divmod(min(p0 + (wave * TY + j) * 32 + l32, last), oh, ow);
    yoff[j] = (oh - oh0) * p.sh * pitch + ow * p.sw * 4 + half * 16;
  }
  v16i acc[TX][TY];
#pragma unroll
  for (int i = 0; i < TX; ++i)
#pragma unroll
    for (int j = 0; j < TY; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  UNIT_WAIT_VMCNT(0);  // the weight fragments have landed
  __syncthreads();

  const int rstep = p.dh * pitch;
  for (int kh = 0; kh < p.KH; ++kh) {
    v4i x[TX], y[TY];
#pragma unroll
    for (int j = 0; j < TY; ++j) y[j] = *reinterpret_cast<const v4i_a4 *>(patch + yoff[j] + kh * rstep);
#pragma unroll
    for (int i = 0; i < TX; ++i) x[i] = *reinterpret_cast<const v4i *>(lds + ((i * p.KH + kh) * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < TX; ++i)
#pragma unroll
      for (int j = 0; j < TY; ++j) acc[i][j] = OpI8::mma(x[i], y[j], acc[i][j]);
  }

  // register r of a lane is channel 8 (r / 4) + 4 half + r % 4 of its pixel: 128 consecutive bytes per 32 lanes
  const __amdgpu_buffer_rsrc_t obuf = result_buffer(p.out);
  const u32 m0 = (u32)(p0 + wave * TY * 32 + l32);
#pragma unroll
  for (int i = 0; i < TX; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c4 = i * 32 + 8 * q + 4 * half;
      const v4i b = *reinterpret_cast<const v4i *>(bias + c4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = kg * (TX * 32) + c4 + e;
        const u32 dst = (u32)(n * p.oc + c) * (u32)p.OHW + m0;
#pragma unroll
        for (int j = 0; j < TY; ++j)
          if (c < p.oc && (int)m0 + j * 32 <= last)
            store_result<kRowPolicy>(obuf, (dst + (u32)(j * 32)) * 4u, (acc[i][j][4 * q + e] + b[e]) * p.scale);
      }
    }
}

// Bytes of LDS of a workgroup of 128 ty pixels and tx channel blocks: the rows that many consecutive pixels can touch.
size_t planar_c4_lds(const ConvGeom &g, int tx, int ty) {
  const int span = (128 * ty + g.OW - 2) / g.OW + 1, rows = (span < g.OH ? span : g.OH) - 1;
  const size_t quads = ((size_t)(g.OW - 1) * g.sw + 8 + 3) / 4;
  return (size_t)tx * (g.KH * 1024 + 128) + ((size_t)rows * g.sh + (size_t)(g.KH - 1) * g.dh + 1) * quads * 16;
}

template <int TX, int TY, int NC>
int launch(const PlanarC4 &p, unsigned grid, size_t lds, hipStream_t s) {
  set_variant("s8stem_nchw_x%d_y%d_c%d", TX * 32, TY * 128, NC);
  hipLaunchKernelGGL((conv_planar_c4_kernel<TX, TY, NC>), dim3(grid), dim3(256), lds, s, p);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK
                         : fail(UNIT_E_LAUNCH, "unit_conv2d_nchw_s8s8s32_fused_prepared: launch: %s", hipGetErrorString(e));
}

template <int TX>
int launch_tx(const PlanarC4 &p, int ty, unsigned grid, size_t lds, hipStream_t s) {
  if (p.C == 3) return ty == 2 ? launch<TX, 2, 3>(p, grid, lds, s) : launch<TX, 1, 3>(p, grid, lds, s);
  return ty == 2 ? launch<TX, 2, 4>(p, grid, lds, s) : launch<TX, 1, 4>(p, grid, lds, s);
}

}  // namespace

// Channel blocks per workgroup: all of them up to three (or a third, half of them), so that no workgroup is partly padding.
static int planar_c4_tx(int kblocks) { return kblocks % 3 == 0 ? 3 : kblocks % 2 == 0 ? 2 : 1; }

// Whether the one-launch kernel takes the convolution: rows of at least a word, and a workgroup's patch and weights in 64 KiB.
bool planar_c4_takes(const ConvGeom &g, int K) {
  return g.W >= 4 && g.c4_steps == g.KH && planar_c4_lds(g, planar_c4_tx((K + 31) / 32), 1) <= 64 * 1024;
}

int conv_planar_c4(const unit_conv_desc *d, const ConvGeom &g, int in_channels, const void *x, const void *w, const int *bias,
                   int scale, void *out, int oc, hipStream_t s) {
  const int kblocks = (d->K + 31) / 32, tx = planar_c4_tx(kblocks), groups = kblocks / tx, ohw = g.OH * g.OW;
  // 256 pixels per workgroup while that leaves two workgroups per CU, else 128
  const int ty = (long)g.N * ceil_div(ohw, 256) * groups >= 512 && planar_c4_lds(g, tx, 2) <= 64 * 1024 ? 2 : 1;
  const int tiles = ceil_div(ohw, 128 * ty);
  PlanarC4 p;
  p.x = static_cast<const char *>(x);
  p.w = static_cast<const char *>(w);
  p.bias = bias;
  p.out = out;
  p.scale = scale;
  p.C = in_channels;
  p.H = g.H;
  p.W = g.W;
  p.OW = g.OW;
  p.OHW = ohw;
  p.KH = g.KH;
  p.sh = g.sh;
  p.sw = g.sw;
  p.dh = g.dh;
  p.pt = g.pt;
  p.pl = g.pl;
  p.oc = oc;
  p.quads = ((g.OW - 1) * g.sw + 8 + 3) / 4;
  p.by_quads = FastDiv::make(p.quads);
  p.by_ow = g.by_ow;
  p.by_tiles = FastDiv::make(tiles);
  p.by_kg = FastDiv::make(groups);
  const unsigned grid = (unsigned)((size_t)g.N * tiles * groups);
  const size_t lds = planar_c4_lds(g, tx, ty);
  switch (tx) {
    case 3: return launch_tx<3>(p, ty, grid, lds, s);
    case 2: return launch_tx<2>(p, ty, grid, lds, s);
    default: return launch_tx<1>(p, ty, grid, lds, s);
  }
}

}  // namespace unit
