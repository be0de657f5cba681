// A network's stem: a 4 x 4 convolution over 16 channels (a 7 x 7 one of stride 2 in
// space-to-depth form), requantized (and clamped), and the 3 x 3 maximum of stride 2 behind it, in
// one launch.
//
// The requantization and the relu do not decrease, so the maximum of the accumulators, requantized,
// is the maximum of the requantized bytes: a quarter of the elements are left to requantize, and
// the convolution's output (51 MB at batch 64, 224 x 224) never reaches memory.
//
// A wave walks down a strip of 14 pooled columns and all (up to 64) channels.  The pixels are the
// rows of the matrix products, so that a lane holds 15 consecutive pixels of one channel: the row
// of a 32 x 32 product that lane group g keeps in register v is pixel 14 g + v, and a row's
// horizontal maxima are seven v_max3 on the lane's own registers.  Pixels outside the image repeat
// the window's nearest one, which a maximum does not notice.  A convolution row shares three of its
// four input rows with the one above, so a wave sends each input row to a ring of seven slots of
// its own in LDS once, four of them on their way, and reads its fragments from there; weights and
// bias stay in registers.  No barrier: nothing but a wave's own rows and the transposition of its
// pooled bytes goes through LDS.
//
// Batch 64, 224 x 224, 3 -> 64 channels: 20.6 us, where the two launches took 27.7 and 15.4.  A
// third of it stays without the products and the requantization: a row is a chain of waiting,
// reading LDS and sending for the next, and two waves a SIMD (the weights of 64 channels in
// registers) cover half of it; one group of 32 channels per wave reads the input twice and is
// level.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_gemm.h"

namespace mxq {
namespace {

#define MXQ_INLINE __attribute__((always_inline))

constexpr int kColumns = 14;  // pooled columns of a wave
constexpr int kAhead = 4;     // input rows on their way beyond the one that is waited for
constexpr int kSlots = 7;     // input rows of a wave in LDS, 2 KB each
constexpr int kPitch = 80;    // bytes of a pooled pixel in LDS

struct StemArgs {
  const int8_t* data;    // [N][H][W][16]
  const int8_t* weight;  // [O][4][4][16]
  int N, H, W, O, ph, pw, OH, OW;
  int PH, PW;            // pooled rows and columns
  int strips, bands, band_rows;  // of an image; pooled rows of a band
  int items;
  Epilogue epi;
};

template <int NI>
__global__ __launch_bounds__(256, 2) void conv_pool_kernel(StemArgs p) {
  constexpr int kStage = kColumns * kPitch;  // bytes of a pooled row
  static_assert(8 * kStage <= NI * 32 * 256 || NI == 1, "the weights' place holds the pooled rows");
  // first the weights, then two pooled rows of each wave
  __shared__ __attribute__((aligned(16))) char shared[NI == 1 ? 8 * kStage : NI * 32 * 256];
  __shared__ __attribute__((aligned(16))) v4i slots[4 * kSlots * 128];
  const int lane = threadIdx.x & 63, lrow = lane & 31, lgrp = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* const stage = shared + wave * 2 * kStage;
  // the last group's idle waves help with the weights, on any item's rows
  const bool idle = blockIdx.x * 4 + wave >= p.items;
  const int item = idle ? 0 : blockIdx.x * 4 + wave;
  const int band = item % p.bands, column = item / p.bands;
  const int strip = column % p.strips, image = column / p.strips;
  const int py0 = band * p.band_rows;
  const int rows = p.PH - py0 < p.band_rows ? p.PH - py0 : p.band_rows;
  const int o0 = blockIdx.y * 32 * NI;

  // the lane's pixel and taps: kw = 2 * pair + lane group
  const int g = (lrow >> 2) & 1, v = (lrow >> 3) * 4 + (lrow & 3);
  int x = 28 * strip - 1 + 14 * g + v;
  x = x < 0 ? 0 : x > p.OW - 1 ? p.OW - 1 : x;
  uint32_t column_at[2];
#pragma unroll
  for (int pair = 0; pair < 2; ++pair) {
    const int ix = x - p.pw + 2 * pair + lgrp;
    column_at[pair] = static_cast<unsigned>(ix) < static_cast<unsigned>(p.W)
                          ? static_cast<uint32_t>(ix) * 16 : kOutOfRange;
  }
  const int8_t* const base = p.data + static_cast<size_t>(image) * p.H * p.W * 16;
  const int first = 2 * py0 - 1;  // convolution row 0 of the walk
  // Input rows come through LDS, a lane's own 16 bytes back into its registers: what is on its way
  // is then counted here (two loads a row, one store every other row, in one order) and not by the
  // compiler, which would have a row wait for the loads that it has just sent wherever a branch
  // lies between.
  const uint32_t slots0 =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(slots)) + wave * kSlots * 2048;
  int sent = 0;  // the slot of the next row that is sent for
  auto send = [&](int i) MXQ_INLINE {
    const int ih = first - p.ph + i;
    const bool in = static_cast<unsigned>(ih) < static_cast<unsigned>(p.H);
    const v4i rsrc = make_rsrc(base + (in ? static_cast<size_t>(ih) * p.W * 16 : 0),
                               in ? static_cast<uint32_t>(p.W) * 16 : 0);
#pragma unroll
    for (int pair = 0; pair < 2; ++pair)
      dma_buffer(__builtin_amdgcn_readfirstlane(slots0 + sent * 2048 + pair * 1024),
                 column_at[pair], rsrc);
    sent = sent + 1 == kSlots ? 0 : sent + 1;
  };
  // What the wave's own lanes wrote to LDS a pooled row ago leaves: LDS executes a wave's
  // instructions in order, so that nothing but the write itself is waited for.  Row -1 of the band
  // and before: nothing, but counted.
  constexpr int PIECES = 2 * NI;
  const int piece_px = lane / PIECES, piece_c = lane % PIECES;
  const int piece_pc = kColumns * strip + piece_px;
  const uint32_t piece_at =
      piece_px < kColumns && piece_pc < p.PW && o0 + piece_c * 16 < p.O
          ? static_cast<uint32_t>(piece_pc * p.O + o0 + piece_c * 16) : kOutOfRange;
  int8_t* const out = p.epi.out8 + (static_cast<size_t>(image) * p.PH + py0) * p.PW * p.O;
  auto store = [&](const char* stage, int k) MXQ_INLINE {
    const bool there = k >= 0 && k < rows;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        out + (there ? static_cast<size_t>(k) * p.PW * p.O : 0), 0, there ? p.PW * p.O : 0,
        0x00020000);
    asm volatile("" ::: "memory");
    const int px = piece_px < kColumns ? piece_px : 0;
    const v4i v = *reinterpret_cast<const v4i*>(stage + px * kPitch + piece_c * 16);
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, piece_at, 0, kDeviceScope);
    asm volatile("" ::: "memory");
  };
  // Everything that the walk starts with goes out at once: the bias, the weights, seven rows (and
  // the stores that a row counts on).  The weights come as the matrix products take them, a
  // channel's 256 bytes over a lane pair, by way of LDS: loaded like that an instruction touches 32
  // lines for 32 bytes of each.
  const EpiScalars s = epi_scalars(p.epi);
  int bias[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int o = o0 + ni * 32 + lrow;
    bias[ni] = o < p.O ? epi_bias32(p.epi, s, o) : 0;
  }
  v4i piece[2 * NI];
  {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.weight), 0,
                                                        p.O * 256, 0x00020000);
#pragma unroll
    for (int i = 0; i < 2 * NI; ++i)
      piece[i] = __builtin_bit_cast(
          v4i, __builtin_amdgcn_raw_buffer_load_b128(
                   rsrc, (o0 + i * 16) * 256 + static_cast<int>(threadIdx.x) * 16, 0, 0));
  }
#pragma unroll
  for (int i = 0; i < 3 + kAhead; ++i) {
    send(i);
    if (i >= 3 && i % 2 == 1) store(stage, -1);
  }
  v4i weight[NI][8];
  {
    v4i* const parked = reinterpret_cast<v4i*>(shared);
#pragma unroll
    for (int i = 0; i < 2 * NI; ++i) {
      const int r = i * 16 + threadIdx.x / 16, c = threadIdx.x % 16;
      parked[r * 16 + (c ^ (r & 15))] = piece[i];
    }
    __syncthreads();
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        weight[ni][ks] = parked[(ni * 32 + lrow) * 16 + ((2 * ks + lgrp) ^ (lrow & 15))];
    __syncthreads();  // the place is the pooled rows' from here on
  }
  bool far = false;  // a sum may wrap around: the bias has to be in it before the maximum is taken
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) far = far || bias[ni] > (1 << 30) || bias[ni] < -(1 << 30);
  far = __any(far);
  const float least = p.epi.relu ? 0.0f : -127.0f;
  wait_vmcnt<0>();
  if (idle) return;
  int taken = 0;  // the slot of the next row that is read
  v4i window[4][2];
  auto take = [&](v4i (&to)[2]) MXQ_INLINE {
    const v4i* const from = slots + (wave * kSlots + taken) * 128 + lane;
    to[0] = from[0];
    to[1] = from[64];
    taken = taken + 1 == kSlots ? 0 : taken + 1;
  };
  take(window[0]);
  take(window[1]);
  take(window[2]);
  // Row 0 sends for the row that takes the first one's slot, and a row outside the image is zeros
  // at once: they must not overtake the read.  (From here on a slot's rows have been multiplied.)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  int above[NI][7];  // the maxima of the window's upper row
  // The horizontal maxima of convolution row r of the walk, R = r mod 4.
  auto maxima = [&](auto at, auto with_bias, int (&most)[NI][7]) MXQ_INLINE {
    constexpr int R = decltype(at)::value;
    v16i acc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      int start = 0;
      if constexpr (decltype(with_bias)::value) {
        start = bias[ni];
        asm volatile("" : "+v"(start));  // 16 copies of it here, not 16 registers for good
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[ni][i] = start;
    }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(window[(R + ks / 2) % 4][ks % 2],
                                                        weight[ni][ks], acc[ni], 0, 0, 0);
    // the first use of a product stays in the block of its last step: with a branch between the
    // two (`if (far) acc += bias`) the wait states come too late and the values are wrong
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        const int a = acc[ni][2 * j], b = acc[ni][2 * j + 1], c = acc[ni][2 * j + 2];
        const int m = a > b ? a : b;
        most[ni][j] = m > c ? m : c;
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto row = [&](auto at, int r, int (&most)[NI][7]) MXQ_INLINE {
    constexpr int R = decltype(at)::value % 4;
    typedef std::integral_constant<int, R> Slot;
    // input row r + 3: the younger ones are kAhead - 1 rows of two loads and kAhead / 2 stores
    wait_vmcnt<2 * (kAhead - 1) + kAhead / 2>();
    take(window[(R + 3) % 4]);
    send(r + 3 + kAhead);
    if (first + r < 0 || first + r >= p.OH) {
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int j = 0; j < 7; ++j) most[ni][j] = INT32_MIN;
    } else if (__builtin_expect(far, 0)) {
      maxima(Slot(), std::true_type(), most);
    } else {
      maxima(Slot(), std::false_type(), most);
    }
  };
  // pooled row k of the band (P = k mod 2), from convolution rows 2 k + 1 and 2 k + 2 of the walk
  auto pooled = [&](auto parity, int k) MXQ_INLINE {
    constexpr int P = decltype(parity)::value;
    int middle[NI][7], below[NI][7];
    row(std::integral_constant<int, 2 * P + 1>(), 2 * k + 1, middle);
    row(std::integral_constant<int, 2 * P + 2>(), 2 * k + 2, below);
    store(stage + (1 - P) * kStage, k - 1);
    char* const to = stage + P * kStage;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        int m = above[ni][j] > middle[ni][j] ? above[ni][j] : middle[ni][j];
        m = m > below[ni][j] ? m : below[ni][j];
        above[ni][j] = below[ni][j];
        if (!far) m += bias[ni];
        to[(7 * lgrp + j) * kPitch + ni * 32 + lrow] =
            static_cast<char>(epi_requant(m, s, least));
      }
  };
  row(std::integral_constant<int, 0>(), 0, above);
  store(stage, -1);
  for (int k = 0; k < rows; k += 2) {
    pooled(std::integral_constant<int, 0>(), k);
    if (k + 1 >= rows) break;
    pooled(std::integral_constant<int, 1>(), k + 1);
  }
  store(stage + (rows - 1) % 2 * kStage, rows - 1);
  wait_vmcnt<0>();  // rows past the band are still on their way to LDS
}

bool conv_pool_ok(int N, int H, int W, int C, int O, int KH, int KW, int ph, int pw, int PH,
                  int PW) {
  if (N <= 0 || C != 16 || KH != 4 || KW != 4 || O <= 0 || O % 16 != 0 || O > 1024) return false;
  if (ph < 0 || pw < 0 || PH <= 0 || PW <= 0) return false;
  const long long OH = 1LL * H + 2 * ph - 3, OW = 1LL * W + 2 * pw - 3;
  if (OH <= 0 || OW <= 0 || OH >= (1LL << 31) || OW >= (1LL << 31)) return false;
  if (1LL * H * W * 16 >= (1LL << 31)) return false;
  // every window holds a pixel
  if (2LL * (PH - 1) - 1 >= OH || 2LL * (PW - 1) - 1 >= OW) return false;
  // offsets in a pooled row, the one that drops a store behind all of them
  if (1LL * PW * O >= (1LL << 31)) return false;
  // two waves a SIMD in bands, or a wave for each strip of every image: 2^32 lanes are a launch's
  const long long strips = 1LL * N * ((PW + kColumns - 1) / kColumns);
  return strips < (1LL << 26) - 4 && strips * PH < (1LL << 29);
}

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" {

int mxq_quantized_conv_pool_fits(int N, int H, int W, int C, int O, int KH, int KW, int pad_h,
                                 int pad_w, int pooled_h, int pooled_w) {
  return conv_pool_ok(N, H, W, C, O, KH, KW, pad_h, pad_w, pooled_h, pooled_w);
}

int mxq_quantized_conv_pool(void* stream, const int8_t* data, const int8_t* weight,
                            const void* prepared, int N, int H, int W, int C, int O, int KH,
                            int KW, int pad_h, int pad_w, int pooled_h, int pooled_w, int8_t* out8,
                            int relu) {
  MXQ_API_BEGIN();
  MXQ_CHECK(conv_pool_ok(N, H, W, C, O, KH, KW, pad_h, pad_w, pooled_h, pooled_w),
            "shape does not qualify for the fused stem");
  MXQ_CHECK(data && weight && prepared && out8, "null pointer");
  MXQ_CHECK(aligned16(data) && aligned16(weight) && aligned16(prepared) && aligned16(out8),
            "unaligned operand");
  StemArgs a = {};
  a.data = data;
  a.weight = weight;
  a.N = N; a.H = H; a.W = W; a.O = O; a.ph = pad_h; a.pw = pad_w;
  a.OH = H + 2 * pad_h - 3;
  a.OW = W + 2 * pad_w - 3;
  a.PH = pooled_h;
  a.PW = pooled_w;
  a.epi.prepared = static_cast<const char*>(prepared);
  a.epi.out8 = out8;
  a.epi.relu = relu;
  a.strips = (pooled_w + kColumns - 1) / kColumns;
  // two waves on every SIMD, and as few rows in common between bands as that leaves
  const long long columns = 1LL * N * a.strips, waves = 8LL * num_cus();
  const long long rows = columns * pooled_h / waves;
  a.band_rows = rows < 1 ? 1 : rows < pooled_h ? static_cast<int>(rows) : pooled_h;
  a.bands = (pooled_h + a.band_rows - 1) / a.band_rows;
  a.items = static_cast<int>(columns * a.bands);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned gx = static_cast<unsigned>((a.items + 3) / 4);
  if (O <= 32)
    hipLaunchKernelGGL((conv_pool_kernel<1>), dim3(gx, 1), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((conv_pool_kernel<2>), dim3(gx, (O + 63) / 64), dim3(256), 0, s, a);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

}  // extern "C"
