// The first convolution of an image network, planar in and out: x (N, C, H, W) s8 with C <= 4, weights in prepared form
// (4-channel blocks), out (N, out_channels, OH, OW) = (conv(x, w) + bias) * scale.  The printed graph runs it as
// layout_transform, convolution, layout_transform (apps/cpu/relay/result.log:6803-6838); here it is one launch.
//
// What bounds it is the result (51 MB at 16 x 3 x 224 x 224, 64 channels, 7 x 7, stride 2: 8 us at the rate of a fill),
// so everything in front of the stores has to be short.  A workgroup takes 128 consecutive output pixels of one
// image and all, a third or half of the channels: it lays the input rows under its window out in LDS, once, as 4-byte pixels with the
// zero padding in place, beside the weight fragments.  A k-step (one window row) is then one 16-byte LDS read per
// 32 pixels -- the direct kernel on a packed copy spends four masked 4-byte gathers from memory there, and a
// launch and a round trip through memory on the copy.  That size: 21.5 us with the packed copy, 13.0 here.
// 128 pixels and not 256: more workgroups than the chip holds at once, so that some load while others store (13.0 against
// 15.4; 32 x 3 x 229 x 92 -> 96, 3 x 3 stride 2, 15.2 against 16.9; one shape of five was 6 % faster on 256).  Results through LDS
// and not 128 bytes per store and channel straight from the accumulators: the latter 18.8 against 15.2, equal on whole lines.
#include "conv_plan.hpp"
#include "conv_prepare.hpp"
#include "mma_dma.hpp"

namespace unit {
namespace {

constexpr int PT = 128;  // output pixels per workgroup

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
template <int TX, int NC>
__global__ __launch_bounds__(256) void conv_planar_c4_kernel(PlanarC4 p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
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

  int oh, ow;
  p.by_ow.divmod(min(p0 + wave * 32 + l32, last), oh, ow);
  const char *window = patch + (oh - oh0) * p.sh * pitch + ow * p.sw * 4 + half * 16;  // its first row, taps 4 half .. + 3
  v16i acc[TX];
#pragma unroll
  for (int i = 0; i < TX; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0;
  UNIT_WAIT_VMCNT(0);  // the weight fragments have landed
  __syncthreads();

  const int rstep = p.dh * pitch;
  for (int kh = 0; kh < p.KH; ++kh) {
    const v4i y = *reinterpret_cast<const v4i_a4 *>(window + kh * rstep);
    v4i x[TX];
#pragma unroll
    for (int i = 0; i < TX; ++i) x[i] = *reinterpret_cast<const v4i *>(lds + ((i * p.KH + kh) * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < TX; ++i) acc[i] = OpI8::mma(x[i], y, acc[i]);
  }

  // Results, 32 channels at a time, through LDS: register r of a lane is channel 8 (r / 4) + 4 half + r % 4 of its pixel;
  // a store instruction then writes 512 consecutive bytes of each of two channel planes.
  v4i add[TX][4];
#pragma unroll
  for (int i = 0; i < TX; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) add[i][q] = *reinterpret_cast<const v4i *>(bias + i * 32 + 8 * q + 4 * half);
  constexpr int kPitch = PT + 4;
  int *tile_out = reinterpret_cast<int *>(lds);
  const __amdgpu_buffer_rsrc_t obuf = result_buffer(p.out);
  const int px = (int)(threadIdx.x * 4) % PT, row0 = (int)(threadIdx.x * 4) / PT;  // eight channels at a time
#pragma unroll
  for (int i = 0; i < TX; ++i) {
    __syncthreads();  // the patch, or the block before, has been read
#pragma unroll
    for (int r = 0; r < 16; ++r)
      tile_out[(8 * (r >> 2) + 4 * half + (r & 3)) * kPitch + wave * 32 + l32] = (acc[i][r] + add[i][r >> 2][r & 3]) * p.scale;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = row0 + k * 8, c = (kg * TX + i) * 32 + row;
      const v4i v = *reinterpret_cast<const v4i *>(tile_out + row * kPitch + px);
      const u32 dst = ((u32)(n * p.oc + c) * (u32)p.OHW + (u32)(p0 + px)) * 4u;
      if (c < p.oc) {
        if (p0 + px + 3 <= last) {
          store_result<kRowPolicy>(obuf, dst, v);
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (p0 + px + e <= last) store_result<kRowPolicy>(obuf, dst + 4u * e, v[e]);
        }
      }
    }
  }
}

// Bytes of the patch: the input rows that PT consecutive pixels can touch.
size_t planar_c4_patch(const ConvGeom &g) {
  const int span = (PT + g.OW - 2) / g.OW + 1, rows = (span < g.OH ? span : g.OH) - 1;
  const size_t quads = ((size_t)(g.OW - 1) * g.sw + 8 + 3) / 4;
  return ((size_t)rows * g.sh + (size_t)(g.KH - 1) * g.dh + 1) * quads * 16;
}

// Bytes of LDS of a workgroup of tx channel blocks: weights, biases and patch, or a block of results.
size_t planar_c4_lds(const ConvGeom &g, int tx) {
  const size_t front = (size_t)tx * (g.KH * 1024 + 128) + planar_c4_patch(g), back = (size_t)32 * (PT + 4) * 4;
  return front > back ? front : back;
}

template <int TX>
int launch(const PlanarC4 &p, unsigned grid, size_t lds, hipStream_t s) {
  const int nc = p.C == 3 ? 3 : 4;
  set_variant("s8stem_nchw_x%d_y%d_c%d", TX * 32, PT, nc);
  hipLaunchKernelGGL((nc == 3 ? conv_planar_c4_kernel<TX, 3> : conv_planar_c4_kernel<TX, 4>), dim3(grid), dim3(256), lds, s, p);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? UNIT_OK
                         : fail(UNIT_E_LAUNCH, "unit_conv2d_nchw_s8s8s32_fused_prepared: launch: %s", hipGetErrorString(e));
}

}  // namespace

// Channel blocks per workgroup: all of them up to three (or a third, half of them), so that no workgroup is partly padding.
static int planar_c4_tx(int kblocks) { return kblocks % 3 == 0 ? 3 : kblocks % 2 == 0 ? 2 : 1; }

// Whether the one-launch kernel takes the convolution: rows of at least a word, and a workgroup's patch and weights in 64 KiB.
// Up to 1024 workgroups, four per CU, it always wins, by the launch it saves.  Past that a workgroup costs about the same
// however many of its 128 pixels exist and however wide the rows are that it lays out for them.  How many pixels may be
// missing goes by what the kernel on a packed copy loses there (us here / there): 1.3 for 1 in general (64 channels, 3 x 3,
// 39062 images of 16 pixels 135 / 32, 9765 of 64 41.6 / 32.8, 4340 of 144 44.3 / 31.2, 1562 of 400 35.3 / 30.8), 1.55 where its
// 64-byte stores do not fit the planes (3698 of 169 45.0 / 53.2), 2 with five or more window rows, a masked gather each there
// (7 x 7, 9765 of 64 49.8 / 55.9, 17361 of 36 81.2 / 60.6), 2.7 where half of its 64-channel tile is padding (32 channels, 25510
// of 49 58.5 / 70.9, 34722 of 36 71.5 / 66.3).  The patch may have 27 KiB (7 x 7 stride 2 on rows of 320 results, 23 KB,
// 44.7 / 47.5, on 384, 28 KB, 48.8 / 47.1, on 640 60.6 / 47.1; 3 x 3 stride 2 on 640, 26 KB, 33.4 / 37.3, on 1024, 41 KB,
// 46.3 / 38.3).
bool planar_c4_takes(const ConvGeom &g, int K) {
  const int kblocks = (K + 31) / 32, tx = planar_c4_tx(kblocks);
  if (g.W < 4 || g.c4_steps != g.KH || planar_c4_lds(g, tx) > 64 * 1024) return false;
  const long pixels = (long)g.OH * g.OW, tiles = (pixels + PT - 1) / PT;
  const int slack = kblocks == 1 ? 270 : g.KH >= 5 ? 200 : pixels % 16 ? 155 : 130;
  return tiles * g.N * (kblocks / tx) <= 1024 || (tiles * PT * 100 <= pixels * slack && planar_c4_patch(g) <= 27 * 1024);
}

int conv_planar_c4(const unit_conv_desc *d, const ConvGeom &g, int in_channels, const void *x, const void *w, const int *bias,
                   int scale, void *out, int oc, hipStream_t s) {
  const int kblocks = (d->K + 31) / 32, tx = planar_c4_tx(kblocks), groups = kblocks / tx, ohw = g.OH * g.OW;
  const int tiles = ceil_div(ohw, PT);
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
  const size_t lds = planar_c4_lds(g, tx);
  switch (tx) {
    case 3: return launch<3>(p, grid, lds, s);
    case 2: return launch<2>(p, grid, lds, s);
    default: return launch<1>(p, grid, lds, s);
  }
}

}  // namespace unit
