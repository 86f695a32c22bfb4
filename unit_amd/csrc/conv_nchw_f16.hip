// The fp16 convolution on plain operands, a (N, C, H, W) and b (K, C, KH, KW), which the reference operator packs
// inside itself (python/tensorizer/ops/gpu.py:25-33): one launch re-lays both operands -- the data as NCHW16c, the
// weights straight into the MFMA fragment order of the prepared kernels -- and a second one convolves.
//
// The re-laying launch is bound by latency at one image and by memory traffic at large batches (it reads and
// writes each operand once).  Packing the weights into the reference's blocked layout first, one thread per element, took
// 4.8 us at 256 x 256 x 3 x 3 and 27 us at 1984 x 496 x 3 x 3 (strided two-byte reads), the data pack another launch of
// 3.4 us, and left the convolution on the per-element weight loads of that layout (10.8 us at 1 x 256 x 30 x 30, stride 2).  That call: 28.1 us then,
// 11.2 us in this form and on the eight-wave tiles that the convolution takes since.
#include "conv_plan.hpp"
#include "conv_prepare.hpp"
#include "mma_core.hpp"

namespace unit {
namespace {

typedef int halves8_t __attribute__((ext_vector_type(4), aligned(2)));  // plain operands may start at any element
constexpr int kMaxWindow = 49;  // positions whose 32 x 16 channel block (1 KiB each) is transposed through LDS

// Workgroups [0, wblocks): weights, one per (32-channel block kb, 16-channel input block ci).  The block's KH * KW
// k-steps are consecutive in the prepared buffer and, per output channel, consecutive in b: rows are read 16 bytes
// per lane into LDS at an odd dword pitch (conflict-free two-byte reads down the 32 rows) and written 1 KiB per wave.
// The other workgroups: data, one pixel x 16 channels per thread (128-byte reads per wave and channel, 2 KiB of
// consecutive output per wave).
__global__ __launch_bounds__(256) void pack_f16_operands(const _Float16 *__restrict__ a, char *__restrict__ packed,
                                                         const _Float16 *__restrict__ b, char *__restrict__ prepared,
                                                         int HW, int cc, size_t npix /* N * cc * HW */, int K, int npos,
                                                         int wblocks, FastDiv by_cc, FastDiv by_hw) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if ((int)blockIdx.x < wblocks) {
    int kb, ci;
    by_cc.divmod((int)blockIdx.x, kb, ci);
    const bool staged = npos <= kMaxWindow;
    const int chunks = 2 * npos, pitch = npos * 32 + 4;  // 16-byte chunks of a row; bytes from row to row in LDS
    const size_t row0 = ((size_t)kb * 32 * cc + ci) * 16 * npos, rstep = (size_t)cc * 16 * npos;
    if (staged) {
      for (int q = threadIdx.x; q < 32 * chunks; q += 256) {
        const int row = q / chunks, ch = q - row * chunks;
        v4i v = {0, 0, 0, 0};
        if (kb * 32 + row < K) v = (v4i)*reinterpret_cast<const halves8_t *>(b + row0 + row * rstep + ch * 8);
        int *dst = reinterpret_cast<int *>(lds + row * pitch + ch * 16);
#pragma unroll
        for (int d = 0; d < 4; ++d) dst[d] = v[d];
      }
      __syncthreads();
    }
    const int lane = threadIdx.x & 63, row = lane & 31, half = lane >> 5;
    for (int p = threadIdx.x >> 6; p < npos; p += 4) {
      v8h h;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int e = (8 * half + k) * npos + p;  // element of the row: input channel, then window position
        if (staged)
          h[k] = *reinterpret_cast<const _Float16 *>(lds + row * pitch + e * 2);
        else
          h[k] = kb * 32 + row < K ? b[row0 + row * rstep + e] : (_Float16)0;
      }
      *reinterpret_cast<v8h *>(prepared + (((size_t)blockIdx.x * npos + p) * 64 + lane) * 16) = h;
    }
    return;
  }
  const size_t i = (size_t)(blockIdx.x - wblocks) * 256 + threadIdx.x;  // (n * cc + ci) * HW + pixel
  if (i >= npix) return;
  size_t plane;
  int pix;
  if (npix < 0x7fffffffull) {
    int q;
    by_hw.divmod((int)i, q, pix);
    plane = q;
  } else {
    plane = i / HW;
    pix = (int)(i - plane * HW);
  }
  const _Float16 *src = a + plane * 16 * HW + pix;
  v8h lo, hi;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    lo[c] = src[(size_t)c * HW];
    hi[c] = src[(size_t)(c + 8) * HW];
  }
  v8h *dst = reinterpret_cast<v8h *>(packed + i * 32);
  dst[0] = lo;
  dst[1] = hi;
}

struct NchwF16Sizes {
  size_t packed, prepared, total;  // bytes; the prepared weights follow the packed data
};

// Checks the descriptor for everything that the convolution rejects -- the operands are re-laid before it runs -- and
// gives the sizes.  The batch may need slices, an image not.
int nchw_f16_sizes(const char *what, const unit_conv_desc *d, NchwF16Sizes *z) {
  int32_t OH, OW;
  if (int rc = unit_conv_out_hw(d, &OH, &OW)) return rc;
  if (d->cb != 16 || d->C % 16 || d->K % 16)
    return fail(UNIT_E_ARG, "%s: C and K must be multiples of 16 and cb 16 (got %d, %d, %d)", what, d->C, d->K, d->cb);
  if (d->pt || d->pl || d->pb || d->pr) return fail(UNIT_E_ARG, "%s: the operator has no padding argument; pre-pad the data", what);
  if (d->dh != 1 || d->dw != 1) return fail(UNIT_E_ARG, "%s: dilation must be 1", what);
  if (d->H >= 16384 || d->W >= 16384) return fail(UNIT_E_ARG, "%s: spatial extent too large", what);  // the window fits the image
  if (!fits((size_t)d->C * d->H * d->W * 2) || !fits((size_t)d->K * d->C * d->KH * d->KW * 2) || !fits((size_t)OH * OW * d->K * 4))
    return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  z->packed = ((size_t)d->N * d->C * d->H * d->W * 2 + 255) / 256 * 256;
  z->prepared = prepared_layout(d->K, d->C, d->KH, d->KW, 16, 2).total_bytes;
  if (!fits(z->prepared)) return fail(UNIT_E_ARG, "%s: tensor exceeds 2^31-1 bytes", what);
  z->total = z->packed + z->prepared;
  return UNIT_OK;
}

}  // namespace
}  // namespace unit

extern "C" int unit_conv2d_nchw_f16f32_ws_bytes(const unit_conv_desc *d, size_t *bytes) {
  using namespace unit;
  const char *what = "unit_conv2d_nchw_f16f32_ws_bytes";
  if (!d || !bytes) return fail(UNIT_E_ARG, "%s: null pointer", what);
  NchwF16Sizes z;
  if (int rc = nchw_f16_sizes(what, d, &z)) return rc;
  *bytes = z.total;
  return UNIT_OK;
}

extern "C" int unit_conv2d_nchw_f16f32(const unit_conv_desc *d, const void *a, const void *b, void *out, void *workspace,
                                       size_t workspace_bytes, unit_stream_t stream) {
  using namespace unit;
  const char *what = "unit_conv2d_nchw_f16f32";
  if (!d || !a || !b || !out || !workspace) return fail(UNIT_E_ARG, "%s: null pointer", what);
  NchwF16Sizes z;
  if (int rc = nchw_f16_sizes(what, d, &z)) return rc;
  if (workspace_bytes < z.total)
    return fail(UNIT_E_ARG, "%s: workspace of %zu bytes needed (got %zu)", what, z.total, workspace_bytes);
  if (int rc = check_aligned(what, {out, workspace})) return rc;
  const int cc = d->C / 16, HW = d->H * d->W, npos = d->KH * d->KW;
  const size_t npix = (size_t)d->N * cc * HW;
  const int wblocks = ceil_div(d->K, 32) * cc;
  const size_t blocks = wblocks + (npix + 255) / 256;
  if (blocks >= 1u << 24) return fail(UNIT_E_ARG, "%s: tensor too large", what);  // a grid has fewer than 2^32 threads
  if (int rc = check_device()) return rc;
  char *packed = static_cast<char *>(workspace), *prepared = packed + z.packed;
  const int lds = npos <= kMaxWindow ? 32 * (npos * 32 + 4) : 0;
  hipLaunchKernelGGL(pack_f16_operands, dim3((unsigned)blocks), dim3(256), lds, static_cast<hipStream_t>(stream),
                     static_cast<const _Float16 *>(a), packed, static_cast<const _Float16 *>(b), prepared, HW, cc, npix, d->K,
                     npos, wblocks, FastDiv::make(cc), FastDiv::make(HW));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UNIT_E_LAUNCH, "%s: launch: %s", what, hipGetErrorString(e));
  return unit_conv2d_nchw16c_f16f32_prepared(d, packed, prepared, out, stream);
}
