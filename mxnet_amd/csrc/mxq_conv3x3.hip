// 3 x 3 convolutions of stride 1 and padding 1 over 256 channels and more, a layer of a plan: its
// weights laid out once as the operands a wave consumes, its scales prepared.
//
// A 7 x 7 plane over 512 channels has 4608 bytes of reduction for each of few pixels.  As tiles
// of an implicit GEMM every 256 bytes of it are a stage that both operands come through LDS for,
// and a barrier: 19 us at batch 64, of which the products are 6.  Here a work-group of eight
// waves takes 64 pixels in memory order by 128 columns.  The pixels its taps touch are one
// contiguous run, a row and a pixel longer on either side, and go to LDS once (42 KB); weights
// come from memory straight into registers, a contiguous KB per step, eight of them on their way;
// and no barrier stands between the first product and the last.  Pixels outside the image are a
// pixel of zeros behind the run.  Two waves share a column tile, each over half of the channels:
// half the weights per wave and two waves a SIMD; their sums meet in LDS at the end, each
// finishing 32 of the pixels.
//
// Bound by the weights' way into a CU (590 KB a group) beside the products.  7 x 7 x 512 -> 512
// in a ResNet-50 at batch 64: 19.0 us -> 11.8.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_forms.h"
#include "mxq_gemm.h"

namespace mxq {
namespace {

#define MXQ_INLINE __attribute__((always_inline))

constexpr int kRows = 64, kColumns = 128;
constexpr int kPitch = kColumns + 16;                    // of an output row in LDS
constexpr int kExchange = 8 * 4096;                      // sums on their way between waves
constexpr int kLeast = kExchange + kRows * kPitch;       // bytes of LDS the end needs

// n / d for n * d < 2^30, magic = 2^31 / d + 1
__device__ __forceinline__ int quotient(int n, uint32_t magic) {
  return static_cast<int>(__umulhi(2u * static_cast<uint32_t>(n) + 1u, magic));
}

struct Conv3x3Args {
  const int8_t* data;     // [M][C]
  const int8_t* weights;  // fragments: [O / 32][9][C / 32] KB
  const char* prepared;
  int8_t* out;            // [M][O]
  int M, H, W, C, O, relu;
  int pixels;             // of the run in LDS, and one of zeros
  uint32_t magic_slots;   // 16-byte slots of a pixel in LDS: one more than its chunks, against banks
};

// G: steps whose weights are on their way
template <int G>
__global__ __launch_bounds__(512, 2) void conv3x3_kernel(Conv3x3Args p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, lrow = lane & 31, lgrp = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ct = wave & 3, kh = wave >> 2;  // column tile, half of the channels
  const int m0 = blockIdx.x * kRows, n0 = blockIdx.y * kColumns;
  const int CH = p.C >> 4, slots = CH + 1, lead = p.W + 1;
  const int per_tap = p.C >> 5, mine = per_tap >> 1;  // steps of a tap, and of this wave

  // the first weights, then the pixels
  const bool has = n0 + ct * 32 < p.O;
  const int column_tiles = (p.O + 31) >> 5;
  const auto weights = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(p.weights), 0, column_tiles * 9 * per_tap * 1024, 0x00020000);
  const int first = (has ? (n0 >> 5) + ct : 0) * 9 * per_tap + kh * mine;
  auto fragment = [&](int k) MXQ_INLINE {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                       weights, lane * 16, k * 1024, 0));
  };
  v4i w[G];
#pragma unroll
  for (int i = 0; i < G; ++i) w[i] = fragment(first + i);
  {
    const v4i rsrc = make_rsrc(p.data, static_cast<uint32_t>(p.M) * p.C);
    const uint32_t at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    const int instructions = (p.pixels * slots + 63) / 64;
    for (int it = wave; it < instructions; it += 8) {
      const int slot = it * 64 + lane, i = quotient(slot, p.magic_slots), c = slot - i * slots;
      const int m = m0 - lead + i;
      const bool in = c < CH && i < p.pixels - 1 && m >= 0 && m < p.M;
      dma_buffer(__builtin_amdgcn_readfirstlane(at + it * 1024),
                 in ? static_cast<uint32_t>(m) * p.C + c * 16 : kOutOfRange, rsrc);
    }
  }
  const EpiScalars s = *reinterpret_cast<const EpiScalars*>(p.prepared);
  const LayerForms forms = *reinterpret_cast<const LayerForms*>(p.prepared + kFormsAt);
  // the lane's two pixels; rows past the end repeat the last one
  int home[2], oh[2], ow[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    int m = m0 + rt * 32 + lrow;
    m = m < p.M ? m : p.M - 1;
    const int rem = m % (p.H * p.W);
    oh[rt] = rem / p.W;
    ow[rt] = rem - oh[rt] * p.W;
    home[rt] = m - m0 + lead;
  }
  auto pixels_under = [&](int tap, int (&at)[2]) MXQ_INLINE {
    const int dh = tap / 3 - 1, dw = tap - 3 * (dh + 1) - 1;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const bool in = static_cast<unsigned>(oh[rt] + dh) < static_cast<unsigned>(p.H) &&
                      static_cast<unsigned>(ow[rt] + dw) < static_cast<unsigned>(p.W);
      at[rt] = ((in ? home[rt] + dh * p.W + dw : p.pixels - 1) * slots + kh * 2 * mine + lgrp) * 16;
    }
  };
  // the accumulators of one half start at the bias
  v16i acc[2];
  {
    const int* const bias = reinterpret_cast<const int*>(p.prepared + kPreparedBias);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int n = n0 + ct * 32 + 8 * (v / 4) + 4 * lgrp + v % 4;
      const int b = kh == 0 && n < p.O ? bias[n] : 0;
      acc[0][v] = b;
      acc[1][v] = b;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

  auto read = [&](v4i (&x)[2], const int (&at)[2], int step) MXQ_INLINE {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
      x[rt] = *reinterpret_cast<const v4i*>(smem + at[rt] + step * 32);
  };
  int now[2], next[2];
  v4i x[2][2];
  pixels_under(0, now);
  read(x[0], now, 0);
  const int groups = mine / G;
  for (int tap = 0; tap < 9; ++tap) {
    pixels_under(tap < 8 ? tap + 1 : 8, next);
    for (int g = 0; g < groups; ++g) {
      const bool last = g + 1 == groups;
      // where the next group's weights lie; past the last one the first ones again
      const int from = last ? (tap < 8 ? first + (tap + 1) * per_tap : first)
                            : first + tap * per_tap + (g + 1) * G;
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (i + 1 < G) {
          read(x[(i + 1) & 1], now, g * G + i + 1);
        } else {
          int at[2];
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) at[rt] = last ? next[rt] : now[rt] + (g + 1) * G * 32;
          read(x[(i + 1) & 1], at, 0);
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
          acc[rt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[i], x[i & 1][rt], acc[rt], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) asm volatile("" : "+v"(acc[rt]));
        w[i] = fragment(from + i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) now[rt] = next[rt];
  }
  // the last products' wait states, before any branch
  asm volatile("s_nop 15\n\ts_nop 15" : "+v"(acc[0]), "+v"(acc[1]));
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the pixels are done with

  // each wave sends what the other of its column tile finishes
  {
    v4i* const to = reinterpret_cast<v4i*>(smem + wave * 4096) + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v4i v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = kh == 0 ? acc[1][4 * i + j] : acc[0][4 * i + j];
      to[i * 64] = v;
    }
  }
  v16i sum;
#pragma unroll
  for (int i = 0; i < 16; ++i) sum[i] = kh == 0 ? acc[0][i] : acc[1][i];
  __syncthreads();
  {
    const v4i* const from = reinterpret_cast<const v4i*>(smem + (wave ^ 4) * 4096) + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4i v = from[i * 64];
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[4 * i + j] += v[j];
    }
  }
  char* const tile = smem + kExchange;
  auto finish = [&](auto pack) MXQ_INLINE {
#pragma unroll
    for (int vq = 0; vq < 4; ++vq)
      *reinterpret_cast<uint32_t*>(tile + (kh * 32 + lrow) * kPitch + ct * 32 + 8 * vq + 4 * lgrp) =
          pack(sum[4 * vq], sum[4 * vq + 1], sum[4 * vq + 2], sum[4 * vq + 3]);
  };
  if (p.relu && (forms.has & 1))
    finish([&](int a, int b, int c, int d) {
      return short_relu4(a, b, c, d, forms.t_relu, forms.c_relu);
    });
  else if (p.relu)
    finish([&](int a, int b, int c, int d) { return epi_requant_pack<true>(a, b, c, d, s); });
  else if (forms.has & 2)
    finish([&](int a, int b, int c, int d) { return short_plain4(a, b, c, d, forms.t_plain); });
  else
    finish([&](int a, int b, int c, int d) { return epi_requant_pack<false>(a, b, c, d, s); });
  __syncthreads();
  const int row = tid >> 3, c = tid & 7;
  if (m0 + row < p.M && n0 + c * 16 < p.O)
    *reinterpret_cast<v4i*>(p.out + static_cast<size_t>(m0 + row) * p.O + n0 + c * 16) =
        *reinterpret_cast<const v4i*>(tile + row * kPitch + c * 16);
}

// [O][9][C] -> fragments [ceil(O / 32)][9][C / 32][64 lanes][16 bytes]: lane l of a step holds bytes
// 16 * (l / 32) ... + 15 of its 32 channels of row l % 32 of the column tile, zeros past the last row.
__global__ __launch_bounds__(256) void pack_conv3x3_kernel(const v4i* in, v4i* out, int O, int CH,
                                                           unsigned pieces) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const int lane = i & 63, steps = CH / 2;
  const unsigned f = i >> 6, t = f / (9 * steps), k = f - t * 9 * steps;
  const int n = 32 * t + (lane & 31);
  out[i] = n < O ? in[static_cast<size_t>(n) * 9 * CH + 2 * k + (lane >> 5)] : v4i{0, 0, 0, 0};
}

bool conv3x3_ok(int N, int H, int W, int C, int O) {
  if (N <= 0 || H <= 0 || W <= 0 || C <= 0 || C % 256 != 0 || O <= 0 || O % 16 != 0) return false;
  const long long M = 1LL * N * H * W, pixels = kRows + 2LL * (W + 1) + 1;
  return M * C < (1LL << 31) && M * O < (1LL << 31) && 9LL * C * ((O + 31) / 32 * 32) < (1LL << 30) &&
         pixels * (C + 16) <= 150 * 1024 && O <= 65535 * kColumns;
}

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" {

// Whether it is also the faster way.  A group alone takes 9 us over 512 channels however few there
// are, where the general path splits few tiles' reduction; from two groups a CU on the weights that
// each group fetches for itself cost what the general path's barriers do.  us, general -> here:
//   7 x 7 x 512 -> 512, by batch: 4  7.4 -> 9.3, 8  8.9 -> 9.3 (28 groups), 16  14.6 -> 9.5 (52),
//     32  14.4 -> 9.6, 64  17.0 -> 11.9, 96  29.7 -> 17.9, 128  33.5 -> 21.3 (392), 256  38.4 -> 38.1
//   14 x 14 x 256 -> 256: 1  4.3 -> 7.1, 8  9.3 -> 7.3 (50), 32  10.8 -> 8.0, 64  14.8 -> 13.9 (392),
//     128  21.8 -> 23.2
//   7 x 7, batch 64: 1024 -> 1024  58.8 -> 38.3, 512 -> 128  14.4 -> 9.4 (49 groups)
// Fewer than 64 columns leave two waves of four without any: 28 x 28 x 256 -> 32  17.4 -> 22.2.
int mxq_quantized_conv3x3_fits(int N, int H, int W, int C, int O) {
  if (!conv3x3_ok(N, H, W, C, O) || O < 64) return 0;
  const long long rows = (1LL * N * H * W + kRows - 1) / kRows;
  const long long groups = rows * ((O + kColumns - 1) / kColumns);
  try {
    return 6 * groups >= num_cus() && groups <= 2 * num_cus();
  } catch (...) {  // no device to ask
    return 0;
  }
}

size_t mxq_quantized_conv3x3_weights(int C, int O) {
  return static_cast<size_t>((O + 31) / 32) * 9 * (C / 32) * 1024;
}

int mxq_pack_conv3x3_weights(void* stream, const int8_t* in, int C, int O, int8_t* out) {
  MXQ_API_BEGIN();
  MXQ_CHECK(conv3x3_ok(1, 1, 1, C, O), "bad channel counts");
  MXQ_CHECK(in && out && aligned16(in) && aligned16(out), "null or unaligned pointer");
  const unsigned pieces = static_cast<unsigned>(mxq_quantized_conv3x3_weights(C, O) / 16);
  hipLaunchKernelGGL(pack_conv3x3_kernel, dim3((pieces + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), reinterpret_cast<const v4i*>(in),
                     reinterpret_cast<v4i*>(out), O, C / 16, pieces);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_quantized_conv3x3(void* stream, const int8_t* data, const int8_t* weights,
                          const void* prepared, int N, int H, int W, int C, int O, int8_t* out8,
                          int relu) {
  MXQ_API_BEGIN();
  MXQ_CHECK(conv3x3_ok(N, H, W, C, O), "shape does not qualify for the 3x3 kernel");
  MXQ_CHECK(data && weights && prepared && out8, "null pointer");
  MXQ_CHECK(aligned16(data) && aligned16(weights) && aligned16(prepared) && aligned16(out8),
            "unaligned operand");
  Conv3x3Args a = {};
  a.data = data;
  a.weights = weights;
  a.prepared = static_cast<const char*>(prepared);
  a.out = out8;
  a.M = N * H * W;
  a.H = H; a.W = W; a.C = C; a.O = O;
  a.relu = relu;
  a.pixels = kRows + 2 * (W + 1) + 1;
  a.magic_slots = static_cast<uint32_t>((1ULL << 31) / static_cast<unsigned>(C / 16 + 1) + 1);
  // whole load instructions
  size_t lds = (static_cast<size_t>(a.pixels) * (C + 16) + 1023) / 1024 * 1024;
  if (lds < kLeast) lds = kLeast;
  const dim3 grid((a.M + kRows - 1) / kRows, (O + kColumns - 1) / kColumns);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (C % 512 == 0)
    hipLaunchKernelGGL(conv3x3_kernel<8>, grid, dim3(512), lds, s, a);
  else
    hipLaunchKernelGGL(conv3x3_kernel<4>, grid, dim3(512), lds, s, a);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

}  // extern "C"
