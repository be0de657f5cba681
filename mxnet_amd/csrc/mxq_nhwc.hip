// Kernels for callers that keep a network's activations as NHWC int8 with the channels padded
// to a multiple of 16 (zeros): the way in from a float NCHW image, the pooling between the
// layers, the weights' layout and the way back to the operator's NCHW tensors.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_gemm.h"

namespace mxq {
namespace {

constexpr int kThreads = 256;

// trunc(sign(x) * min(|x| * s + 0.5f, 127.f)), quantize_v2-inl.h:66-95
__device__ __forceinline__ uint32_t quant_byte(float x, float s) {
  const float t = fabsf(x) * s + 0.5f;
  const int v = static_cast<int>(127.0f < t ? 127.0f : t);
  return static_cast<uint32_t>(x < 0.0f ? -v : (x > 0.0f ? v : 0)) & 0xffu;
}

struct QuantNhwcArgs {
  const float* in;  // [N][C][H][W]
  v4i* out;         // [N][OH][OW][Cp / 16]
  float* omin;
  float* omax;
  int C, H, W, OH, OW, chunks, off_h, off_w;
  float range;
  size_t pieces;  // 16-byte pieces of the output
};

// One 16-byte piece of one output pixel per lane: consecutive lanes read consecutive pixels of
// each channel plane.  Bound by the float image (38.5 MB at batch 64, 224 x 224).  Against
// quantize_v2 followed by the layout adapter the int8 NCHW tensor between them is neither
// written nor read, and one launch is saved.
// S2D: space to depth by 2 on the way, as mxq_nchw_to_s2d_nhwc_i8.
template <bool S2D>
__global__ __launch_bounds__(kThreads) void quantize_nhwc_kernel(QuantNhwcArgs a) {
  const size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i == 0) {
    *a.omin = -a.range;
    *a.omax = a.range;
  }
  if (i >= a.pieces) return;
  const float s = 127.0f / a.range;
  // pieces of one chunk of an image's pixels are neighbours
  const int plane = a.OH * a.OW;
  const size_t row = i / plane;
  const int pixel = static_cast<int>(i - row * plane);
  const size_t n = row / a.chunks;
  const int chunk = static_cast<int>(row - n * a.chunks);
  const int oh = pixel / a.OW, ow = pixel - oh * a.OW;
  const float* img = a.in + n * a.C * a.H * a.W;
  const size_t stride = static_cast<size_t>(a.H) * a.W;
  uint32_t w[4] = {0, 0, 0, 0};
  if (S2D) {
    int d = chunk * 16 / a.C, c = chunk * 16 - d * a.C;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int h = 2 * oh - a.off_h + (d >> 1), x = 2 * ow - a.off_w + (d & 1);
      if (d < 4 && static_cast<unsigned>(h) < static_cast<unsigned>(a.H) &&
          static_cast<unsigned>(x) < static_cast<unsigned>(a.W))
        w[k >> 2] |= quant_byte(img[c * stride + static_cast<size_t>(h) * a.W + x], s)
                     << (8 * (k & 3));
      if (++c == a.C) {
        c = 0;
        ++d;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int c = chunk * 16 + k;
      if (c < a.C) w[k >> 2] |= quant_byte(img[c * stride + pixel], s) << (8 * (k & 3));
    }
  }
  a.out[(n * plane + pixel) * a.chunks + chunk] =
      v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]),
          static_cast<int>(w[3])};
}

// The same for an image of up to four channels in space-to-depth form, a pixel of 16 bytes per lane:
// two neighbouring columns of each channel and row, loaded as one, all of them before the first is
// looked at (clamped into the image and taken out again where they were outside).  224 x 224 x 3
// in the head of a network's pass: batch 64 9.9 us, one image 3.2 (with the channels a variable and
// a branch around each load 13.4 and 6.7).
// PAIR: images of two columns and more.  FLAT: lanes run on from one image to the next, for planes
// that leave much of a work-group's last lanes idle (60000 images of 3 x 4 x 4 29.4 us -> 6.4, 8000 of
// 8 x 8 6.2 -> 3.6, 200 of 3 x 40 x 40 3.3 -> 3.2); else images are the grid's second axis, which saves
// a division.
constexpr int kS2dThreads = 128;
constexpr int kS2dFlat = 1024;  // pixels of a plane from which on images are an axis
template <int C, bool PAIR, bool FLAT>
__global__ __launch_bounds__(kS2dThreads) void quantize_s2d_kernel(QuantNhwcArgs a) {
  const int plane = a.OH * a.OW;
  unsigned at = blockIdx.x * kS2dThreads + threadIdx.x, image = blockIdx.y;
  if (at == 0 && image == 0) {
    *a.omin = -a.range;
    *a.omax = a.range;
  }
  if (FLAT) {
    if (at >= a.pieces) return;
    image = at / static_cast<unsigned>(plane);
    at -= image * static_cast<unsigned>(plane);
  } else if (at >= static_cast<unsigned>(plane)) {
    return;
  }
  const int pixel = static_cast<int>(at);
  const float s = 127.0f / a.range;
  const int oh = static_cast<int>(static_cast<unsigned>(pixel) / static_cast<unsigned>(a.OW));
  const int x = 2 * (pixel - oh * a.OW) - a.off_w, y = 2 * oh - a.off_h;
  const int from = !PAIR || x < 0 ? 0 : x > a.W - 2 ? a.W - 2 : x;
  const float* const img = a.in + static_cast<size_t>(image) * C * a.H * a.W;
  float v[2][C][2] = {};
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int h = y + d < 0 ? 0 : y + d > a.H - 1 ? a.H - 1 : y + d;
#pragma unroll
    for (int c = 0; c < C; ++c)
      __builtin_memcpy(v[d][c], img + (static_cast<size_t>(c) * a.H + h) * a.W + from, PAIR ? 8 : 4);
  }
  int q[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) q[k] = 0;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const bool row = static_cast<unsigned>(y + d) < static_cast<unsigned>(a.H);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const bool in = row && static_cast<unsigned>(x + e) < static_cast<unsigned>(a.W);
      const bool high = x + e != from;  // of the pair
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const float f = in ? (high ? v[d][c][1] : v[d][c][0]) : 0.0f;
        const float t = fabsf(f) * s + 0.5f;
        // the sign before the conversion: it truncates either side alike
        q[(2 * d + e) * C + c] = static_cast<int>(copysignf(127.0f < t ? 127.0f : t, f));
      }
    }
  }
  v4i w;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w[j] = static_cast<int>(pack_bytes(q[4 * j], q[4 * j + 1], q[4 * j + 2], q[4 * j + 3]));
  a.out[static_cast<size_t>(image) * plane + pixel] = w;
}

struct PoolNhwcArgs {
  const v4i* in;  // [N][H][W][chunks]
  v4i* out;       // [N][OH][OW][chunks]
  int H, W, OH, OW, KH, KW, sh, sw, ph, pw, chunks, count_pad;
  int outputs;    // N * OH * OW
  size_t pieces;  // outputs * chunks
};

typedef short s2 __attribute__((ext_vector_type(2)));

// maximum of the four int8 of each dword: as two pairs of 16-bit values whose upper byte is the
// int8 (v_pk_max_i16)
__device__ __forceinline__ void max_bytes(uint32_t x, s2& even, s2& odd) {
  const s2 e = __builtin_bit_cast(s2, (x << 8) & 0xff00ff00u);
  const s2 o = __builtin_bit_cast(s2, x & 0xff00ff00u);
  even = __builtin_elementwise_max(even, e);
  odd = __builtin_elementwise_max(odd, o);
}

struct Window {
  int h0, h1, w0, w1, divisor;
};
// the window inside the image, and the divisor of an average (src/operator/nn/pool.h:476-522)
__device__ __forceinline__ Window window_of(const PoolNhwcArgs& a, int oh, int ow) {
  Window r;
  r.h0 = oh * a.sh - a.ph;
  r.w0 = ow * a.sw - a.pw;
  r.h1 = min(r.h0 + a.KH, a.H + a.ph);
  r.w1 = min(r.w0 + a.KW, a.W + a.pw);
  r.divisor = (r.h1 - r.h0) * (r.w1 - r.w0);
  r.h0 = max(r.h0, 0);
  r.w0 = max(r.w0, 0);
  // a window that misses the image is empty in that direction: callers multiply the two extents
  r.h1 = max(min(r.h1, a.H), r.h0);
  r.w1 = max(min(r.w1, a.W), r.w0);
  if (!a.count_pad) r.divisor = (r.h1 - r.h0) * (r.w1 - r.w0);
  return r;
}
__device__ __forceinline__ uint32_t average_byte(int sum, int divisor) {
  // nearest, ties to even (the binary32 quotient is exact on ties and cannot round onto one)
  const float avg = divisor > 0 ? static_cast<float>(sum) / static_cast<float>(divisor) : 0.f;
  return static_cast<uint32_t>(min(max(static_cast<int>(rintf(avg)), -128), 127)) & 0xffu;
}
__device__ __forceinline__ int byte_at(v4i v, int k) {
  return static_cast<int8_t>((static_cast<uint32_t>(v[k >> 2]) >> (8 * (k & 3))) & 0xffu);
}

// One 16-byte piece of an output pixel per lane; the lanes of a wave read whole pixels.  The
// rows of neighbouring windows meet in L1 / L2, so the input crosses HBM once.
template <bool AVG>
__global__ __launch_bounds__(kThreads) void pool_nhwc_kernel(PoolNhwcArgs a) {
  const size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= a.pieces) return;
  const int o = static_cast<int>(i / a.chunks);
  const int chunk = static_cast<int>(i - static_cast<size_t>(o) * a.chunks);
  const int t = o / a.OW, ow = o - t * a.OW;
  const int n = t / a.OH, oh = t - n * a.OH;
  const Window win = window_of(a, oh, ow);
  const v4i* img = a.in + static_cast<size_t>(n) * a.H * a.W * a.chunks + chunk;
  v4i out;
  if (AVG) {
    int sum[16] = {};
    for (int h = win.h0; h < win.h1; ++h)
      for (int w = win.w0; w < win.w1; ++w) {
        const v4i v = img[(static_cast<size_t>(h) * a.W + w) * a.chunks];
#pragma unroll
        for (int k = 0; k < 16; ++k) sum[k] += byte_at(v, k);
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) w |= average_byte(sum[4 * q + k], win.divisor) << (8 * k);
      out[q] = static_cast<int>(w);
    }
  } else {
    s2 even[4], odd[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) even[q] = odd[q] = s2{-32768, -32768};
    for (int h = win.h0; h < win.h1; ++h)
      for (int w = win.w0; w < win.w1; ++w) {
        const v4i v = img[(static_cast<size_t>(h) * a.W + w) * a.chunks];
#pragma unroll
        for (int q = 0; q < 4; ++q) max_bytes(static_cast<uint32_t>(v[q]), even[q], odd[q]);
      }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      out[q] = static_cast<int>((__builtin_bit_cast(uint32_t, even[q]) >> 8) |
                                __builtin_bit_cast(uint32_t, odd[q]));
  }
  a.out[i] = out;
}

// The maximum over 3 x 3 windows (a network's stem).  With the window's extents known all nine
// loads are on their way at once; a row or column outside the image reads the window's nearest one
// again, which a maximum does not notice.
__global__ __launch_bounds__(kThreads) void max3x3_nhwc_kernel(PoolNhwcArgs a) {
  const size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= a.pieces) return;
  const int o = static_cast<int>(i / a.chunks);
  const int chunk = static_cast<int>(i - static_cast<size_t>(o) * a.chunks);
  const int t = o / a.OW, ow = o - t * a.OW;
  const int n = t / a.OH, oh = t - n * a.OH;
  const Window win = window_of(a, oh, ow);
  v4i out;
  if (win.h0 < win.h1 && win.w0 < win.w1) {
    const v4i* img = a.in + static_cast<size_t>(n) * a.H * a.W * a.chunks + chunk;
    v4i v[9];
#pragma unroll
    for (int h = 0; h < 3; ++h)
#pragma unroll
      for (int w = 0; w < 3; ++w)
        v[3 * h + w] = img[(static_cast<size_t>(min(win.h0 + h, win.h1 - 1)) * a.W +
                            min(win.w0 + w, win.w1 - 1)) * a.chunks];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s2 even = s2{-32768, -32768}, odd = even;
#pragma unroll
      for (int k = 0; k < 9; ++k) max_bytes(static_cast<uint32_t>(v[k][q]), even, odd);
      out[q] = static_cast<int>((__builtin_bit_cast(uint32_t, even) >> 8) |
                                __builtin_bit_cast(uint32_t, odd));
    }
  } else {
    out = v4i{1, 1, 1, 1} * static_cast<int>(0x80808080u);
  }
  a.out[i] = out;
}

// Averages over large windows (global pooling: one window per image and channel): 16 lanes take
// 16 pieces of a pixel, 16 such groups the pixels of the window in turn, and the 16 partial sums
// meet in LDS.  One lane walking a 7 x 7 window alone is 49 dependent round trips to memory.
__global__ __launch_bounds__(kThreads) void pool_nhwc_wide_kernel(PoolNhwcArgs a) {
  __shared__ int part[16][16][17];
  const int lane = threadIdx.x & 15, group = threadIdx.x >> 4;
  const int blocks_per_output = (a.chunks + 15) / 16;
  const int o = blockIdx.x / blocks_per_output;
  const int chunk = (blockIdx.x - o * blocks_per_output) * 16 + lane;
  const int t = o / a.OW, ow = o - t * a.OW;
  const int n = t / a.OH, oh = t - n * a.OH;
  const Window win = window_of(a, oh, ow);
  int sum[16] = {};
  if (chunk < a.chunks) {
    const v4i* img = a.in + static_cast<size_t>(n) * a.H * a.W * a.chunks + chunk;
    const int across = win.w1 - win.w0, count = (win.h1 - win.h0) * across;
    for (int p = group; p < count; p += 16) {
      const int h = win.h0 + p / across, w = win.w0 + p % across;
      const v4i v = img[(static_cast<size_t>(h) * a.W + w) * a.chunks];
#pragma unroll
      for (int k = 0; k < 16; ++k) sum[k] += byte_at(v, k);
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) part[group][lane][k] = sum[k];
  __syncthreads();
  // thread (lane, group): channel `group` of piece `lane`
  int total = 0;
#pragma unroll
  for (int g = 0; g < 16; ++g) total += part[g][lane][group];
  if (chunk < a.chunks)
    reinterpret_cast<uint8_t*>(a.out + static_cast<size_t>(o) * a.chunks + chunk)[group] =
        static_cast<uint8_t>(average_byte(total, win.divisor));
}

struct PackArgs {
  const int8_t* in;  // [O][C][KH][KW]
  int8_t* out;       // [Op][OKH][OKW][Cp]
  int O, C, KH, KW, OKH, OKW, Cp;
  size_t bytes;      // of the output
};

// Once per weight tensor: one byte per lane.
template <bool S2D>
__global__ __launch_bounds__(kThreads) void pack_weight_kernel(PackArgs a) {
  const size_t stride = size_t(gridDim.x) * kThreads;
  for (size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x; i < a.bytes; i += stride) {
    size_t t = i / a.Cp;
    const int k = static_cast<int>(i - t * a.Cp);
    const size_t t2 = t / a.OKW;
    int kw = static_cast<int>(t - t2 * a.OKW);
    const size_t o = t2 / a.OKH;
    int kh = static_cast<int>(t2 - o * a.OKH);
    int c = k;
    bool ok = o < static_cast<size_t>(a.O);
    if (S2D) {
      const int d = k / a.C;
      c = k - d * a.C;
      kh = 2 * kh + (d >> 1);
      kw = 2 * kw + (d & 1);
      ok = ok && d < 4;
    }
    ok = ok && c < a.C && kh < a.KH && kw < a.KW;
    a.out[i] = ok ? a.in[((o * a.C + c) * a.KH + kh) * a.KW + kw] : int8_t(0);
  }
}

// [N][HW][Cp] -> [N][C][HW]: a rarely taken way out, one byte per lane
__global__ __launch_bounds__(kThreads) void unpad_kernel(const int8_t* in, int8_t* out, int C,
                                                         int HW, int Cp, size_t bytes) {
  const size_t stride = size_t(gridDim.x) * kThreads;
  for (size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x; i < bytes; i += stride) {
    const size_t t = i / HW;
    const int p = static_cast<int>(i - t * HW);
    const size_t n = t / C;
    const int c = static_cast<int>(t - n * C);
    out[i] = in[(n * HW + p) * Cp + c];
  }
}

unsigned blocks_for(size_t items) {
  const size_t g = (items + kThreads - 1) / kThreads;
  MXQ_CHECK(g < (size_t(1) << 31), "tensor too large for one launch");
  return static_cast<unsigned>(g);
}

unsigned capped_blocks(size_t items) {
  const size_t cap = static_cast<size_t>(num_cus()) * 16;
  const size_t g = (items + kThreads - 1) / kThreads;
  return static_cast<unsigned>(g < cap ? g : cap);
}

// Images in as many launches as their lanes (FLAT) or the grid's second axis need.
template <int C, bool PAIR, bool FLAT>
void launch_s2d_as(hipStream_t s, QuantNhwcArgs a, int N) {
  const long long plane = 1LL * a.OH * a.OW;  // up to the last int
  const int most = FLAT ? static_cast<int>(((1LL << 31) - 1) / plane) : 65535;
  for (int left = N; left > 0; left -= most) {
    const int images = left < most ? left : most;
    a.pieces = static_cast<size_t>(images) * plane;
    const long long lanes = FLAT ? images * plane : plane;
    const dim3 grid(static_cast<unsigned>((lanes + kS2dThreads - 1) / kS2dThreads),
                    FLAT ? 1 : images);
    hipLaunchKernelGGL((quantize_s2d_kernel<C, PAIR, FLAT>), grid, dim3(kS2dThreads), 0, s, a);
    MXQ_LAUNCH_CHECK();
    a.in += static_cast<size_t>(images) * a.C * a.H * a.W;
    a.out += a.pieces;
  }
}
template <int C>
void launch_s2d(hipStream_t s, const QuantNhwcArgs& a, int N) {
  const bool flat = 1LL * a.OH * a.OW < kS2dFlat;
  if (a.W == 1)
    flat ? launch_s2d_as<C, false, true>(s, a, N) : launch_s2d_as<C, false, false>(s, a, N);
  else
    flat ? launch_s2d_as<C, true, true>(s, a, N) : launch_s2d_as<C, true, false>(s, a, N);
}

// One row or column of the space-to-depth form more than the image has: `more_h`, `more_w`.
void quantize_to_nhwc(void* stream, const float* in, int8_t* out, float* omin, float* omax, int N,
                      int C, int H, int W, int C_padded, bool space_to_depth, int off_h, int off_w,
                      int more_h, int more_w, float min_calib, float max_calib) {
  MXQ_CHECK(N >= 0 && C > 0 && H > 0 && W > 0, "bad shape");
  MXQ_CHECK(C_padded % 16 == 0 && C_padded >= (space_to_depth ? 4 : 1) * C, "bad C_padded");
  MXQ_CHECK((off_h == 0 || off_h == 1) && (off_w == 0 || off_w == 1), "offsets are 0 or 1");
  MXQ_CHECK(omin != nullptr && omax != nullptr, "null range output");
  QuantNhwcArgs a;
  a.in = in;
  a.out = reinterpret_cast<v4i*>(out);
  a.omin = omin;
  a.omax = omax;
  a.C = C; a.H = H; a.W = W;
  a.OH = space_to_depth ? (H + off_h + 1) / 2 + more_h : H;
  a.OW = space_to_depth ? (W + off_w + 1) / 2 + more_w : W;
  a.chunks = C_padded / 16;
  a.off_h = off_h;
  a.off_w = off_w;
  const float x = fabsf(min_calib), y = fabsf(max_calib);
  a.range = (x < y) ? y : x;
  MXQ_CHECK(static_cast<long long>(a.OH) * a.OW < (1LL << 31), "image too large");
  a.pieces = static_cast<size_t>(N) * a.OH * a.OW * a.chunks;
  if (a.pieces == 0) return;
  MXQ_CHECK(in != nullptr && out != nullptr && aligned16(out), "null or unaligned data pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (space_to_depth && C <= 4 && a.chunks == 1) {
    switch (C) {
      case 1: launch_s2d<1>(s, a, N); break;
      case 2: launch_s2d<2>(s, a, N); break;
      case 3: launch_s2d<3>(s, a, N); break;
      default: launch_s2d<4>(s, a, N);
    }
  } else if (space_to_depth)
    hipLaunchKernelGGL((quantize_nhwc_kernel<true>), dim3(blocks_for(a.pieces)), dim3(kThreads),
                       0, s, a);
  else
    hipLaunchKernelGGL((quantize_nhwc_kernel<false>), dim3(blocks_for(a.pieces)), dim3(kThreads),
                       0, s, a);
  MXQ_LAUNCH_CHECK();
}

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" {

int mxq_quantize_to_nhwc(void* stream, const float* in, int8_t* out, float* omin, float* omax,
                         int N, int C, int H, int W, int C_padded, int space_to_depth, int off_h,
                         int off_w, float min_calib, float max_calib) {
  MXQ_API_BEGIN();
  quantize_to_nhwc(stream, in, out, omin, omax, N, C, H, W, C_padded, space_to_depth != 0, off_h,
                   off_w, 0, 0, min_calib, max_calib);
  MXQ_API_END();
}

int mxq_quantize_to_s2d(void* stream, const float* in, int8_t* out, float* omin, float* omax,
                        int N, int C, int H, int W, int C_padded, int off_h, int off_w, int H2,
                        int W2, float min_calib, float max_calib) {
  MXQ_API_BEGIN();
  MXQ_CHECK(H > 0 && W > 0, "bad shape");
  const long long more_h = H2 - (1LL * H + off_h + 1) / 2, more_w = W2 - (1LL * W + off_w + 1) / 2;
  MXQ_CHECK((more_h == 0 || more_h == 1) && (more_w == 0 || more_w == 1),
            "rows and columns that the image does not give");
  quantize_to_nhwc(stream, in, out, omin, omax, N, C, H, W, C_padded, true, off_h, off_w,
                   static_cast<int>(more_h), static_cast<int>(more_w), min_calib, max_calib);
  MXQ_API_END();
}

int mxq_quantized_pooling_nhwc(void* stream, const int8_t* in, int N, int H, int W, int C,
                               int kernel_h, int kernel_w, int stride_h, int stride_w, int pad_h,
                               int pad_w, int OH, int OW, int pool_type, int count_include_pad,
                               int8_t* out) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && H > 0 && W > 0 && C > 0 && C % 16 == 0, "bad shape");
  MXQ_CHECK(kernel_h > 0 && kernel_w > 0 && stride_h > 0 && stride_w > 0 && pad_h >= 0 &&
                pad_w >= 0 && OH > 0 && OW > 0,
            "bad window");
  MXQ_CHECK(pool_type == MXQ_POOL_MAX || pool_type == MXQ_POOL_AVG, "unknown pool_type");
  PoolNhwcArgs a;
  a.in = reinterpret_cast<const v4i*>(in);
  a.out = reinterpret_cast<v4i*>(out);
  a.H = H; a.W = W; a.OH = OH; a.OW = OW; a.KH = kernel_h; a.KW = kernel_w;
  a.sh = stride_h; a.sw = stride_w; a.ph = pad_h; a.pw = pad_w;
  a.chunks = C / 16;
  a.count_pad = count_include_pad != 0;
  MXQ_CHECK(static_cast<long long>(N) * OH * OW < (1LL << 31), "problem too large");
  a.outputs = N * OH * OW;
  a.pieces = static_cast<size_t>(a.outputs) * a.chunks;
  if (a.pieces == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr && aligned16(in) && aligned16(out),
            "null or unaligned data pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // from 16 pixels on a window's loads are spread over lanes
  if (pool_type == MXQ_POOL_AVG && static_cast<long long>(kernel_h) * kernel_w >= 16) {
    const size_t g = static_cast<size_t>(a.outputs) * ((a.chunks + 15) / 16);
    MXQ_CHECK(g < (size_t(1) << 31), "problem too large");
    hipLaunchKernelGGL(pool_nhwc_wide_kernel, dim3(static_cast<unsigned>(g)), dim3(kThreads), 0, s,
                       a);
  } else if (pool_type == MXQ_POOL_AVG) {
    hipLaunchKernelGGL((pool_nhwc_kernel<true>), dim3(blocks_for(a.pieces)), dim3(kThreads), 0, s,
                       a);
  } else if (kernel_h == 3 && kernel_w == 3) {
    hipLaunchKernelGGL(max3x3_nhwc_kernel, dim3(blocks_for(a.pieces)), dim3(kThreads), 0, s, a);
  } else {
    hipLaunchKernelGGL((pool_nhwc_kernel<false>), dim3(blocks_for(a.pieces)), dim3(kThreads), 0,
                       s, a);
  }
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_pack_weight(void* stream, const int8_t* in, int8_t* out, int O, int C, int KH, int KW,
                    int O_padded, int C_padded, int space_to_depth) {
  MXQ_API_BEGIN();
  MXQ_CHECK(O > 0 && C > 0 && KH > 0 && KW > 0, "bad shape");
  MXQ_CHECK(O_padded >= O && C_padded >= (space_to_depth ? 4 : 1) * C, "bad padded extent");
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  PackArgs a;
  a.in = in;
  a.out = out;
  a.O = O; a.C = C; a.KH = KH; a.KW = KW;
  a.OKH = space_to_depth ? (KH + 1) / 2 : KH;
  a.OKW = space_to_depth ? (KW + 1) / 2 : KW;
  a.Cp = C_padded;
  a.bytes = static_cast<size_t>(O_padded) * a.OKH * a.OKW * C_padded;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (space_to_depth)
    hipLaunchKernelGGL((pack_weight_kernel<true>), dim3(capped_blocks(a.bytes)), dim3(kThreads),
                       0, s, a);
  else
    hipLaunchKernelGGL((pack_weight_kernel<false>), dim3(capped_blocks(a.bytes)), dim3(kThreads),
                       0, s, a);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_nhwc_pad_to_nchw_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int C_padded) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && C >= 0 && H >= 0 && W >= 0, "negative dimension");
  MXQ_CHECK(C_padded >= C, "C_padded must be at least C");
  MXQ_CHECK(static_cast<long long>(H) * W < (1LL << 31), "image too large");
  if (C_padded == C) return mxq_nhwc_to_nchw(stream, in, out, N, C, H, W, 1);
  const size_t bytes = static_cast<size_t>(N) * C * H * W;
  if (bytes == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  hipLaunchKernelGGL(unpad_kernel, dim3(capped_blocks(bytes)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), in, out, C, H * W, C_padded, bytes);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

}  // extern "C"
