// Contractions with few output tiles: a fully-connected layer at small batch, a convolution of
// one image.  The tiled kernels walk such a reduction alone, one 64 x 64 tile per work-group and
// a barrier per stage: a 3 x 3 convolution over 512 channels of one 7 x 7 plane is 8 work-groups
// of 18 stages, 15-17 us, nearly all of it waiting for memory.
//
// Here a work-group owns a 32 x 32 or 16 x 16 output tile and its waves share the reduction: wave w takes
// the 128-byte blocks w, w + W, ... of the K axis, loads both operands' fragments straight from
// memory into the MFMA layout (no LDS, no barrier, two or three blocks in flight per wave), and the
// W partial tiles meet in LDS once at the end.  Integer addition is associative: the result is the
// tiled kernels' bit for bit.  The same convolution: 5.4 us, of which an empty launch is 3.0.
//
// Four consecutive lanes load 64 consecutive bytes of one row, which is what the address unit
// handles in one step; the MFMA wants consecutive lanes to hold consecutive rows, so the pieces
// change lanes (ds_bpermute) before they are multiplied.  Loaded in the MFMA's own layout every
// lane of a group of four touches a cache line of its own and a CU takes in 18 bytes per clock
// (49 x 4096 -> 512: 9.4 us).
//
// The operands need no alignment: a row that does not start on a 16-byte mark is read with
// unaligned 16-byte loads and masked at its end.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_few_tiles.h"
#include "mxq_gemm.h"

namespace mxq {
namespace {

constexpr int kBlockK = 128;    // bytes of the reduction a wave takes at a time: a cache line
constexpr int kSteps = kBlockK / 64;
// blocks in flight per wave: three, two where 16 waves leave a lane 128 registers and a block of
// a 32 x 32 tile takes 32 of them
constexpr int depth_of(int waves, int tile) { return waves == 16 && tile == 32 ? 2 : 3; }

// 16-byte pieces of row-major rows of K bytes, aligned: pieces past the row, rows past the
// operand and blocks past the reduction come back as zeros without being fetched.
struct AlignedRows {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t row;  // byte offset of the lane's row, or out of range
  int K;
  __device__ __forceinline__ void init(const int8_t* base, int r, int rows, int k) {
    K = k;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base), 0,
                                             static_cast<uint32_t>(rows) * K, 0x00020000);
    row = r < rows ? static_cast<uint32_t>(r) * K : kOutOfRange;
  }
  __device__ __forceinline__ v4i load(int k0) const {
    const uint32_t off = k0 < K ? row + static_cast<uint32_t>(k0) : kOutOfRange;
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                       rsrc, row == kOutOfRange ? kOutOfRange : off, 0, 0));
  }
};

// The same for any K and base.  A piece that would pass the operand's last byte is read from 16
// bytes before that end and shifted into place.
struct AnyRows {
  const int8_t* base;
  long long row, total;
  int K;
  bool ok;
  __device__ __forceinline__ void init(const int8_t* b, int r, int rows, int k) {
    base = b;
    K = k;
    total = static_cast<long long>(rows) * K;
    ok = r < rows;
    row = ok ? static_cast<long long>(r) * K : 0;
  }
  __device__ __forceinline__ v4i load(int k0) const {
    const int left = ok ? K - k0 : 0;  // bytes of the row from here on
    const long long off = left > 0 ? row + k0 : 0;
    const long long from = off < total - 16 ? off : total - 16;
    v4i v;
    __builtin_memcpy(&v, base + from, 16);
    const int shift = static_cast<int>(off - from);
    if (__builtin_expect(__any(left < 16 || shift != 0), 0)) {
      unsigned __int128 w = __builtin_bit_cast(unsigned __int128, v) >> (8 * shift);
      const int drop = left >= 16 ? 0 : left > 0 ? 16 - left : 16;
      w = drop >= 16 ? 0 : (w << (8 * drop)) >> (8 * drop);
      v = __builtin_bit_cast(v4i, w);
    }
    return v;
  }
};

// floor(n / d) for n * d < 2^32, magic = 2^32 / d + 1 (0 stands for d = 1)
__device__ __forceinline__ int few_tiles_div(int n, uint32_t magic) {
  return magic == 0 ? n : static_cast<int>(__umulhi(static_cast<uint32_t>(n), magic));
}

// Pieces of an NHWC convolution's implicit rows: 16 channels of one tap (16 | C).
struct ConvRows {
  __amdgpu_buffer_rsrc_t rsrc;
  int pix, ih0, iw0, C, W, H, KW, K, dh, dw;
  uint32_t magic_c, magic_kw;
  bool ok;
  __device__ __forceinline__ void init(const FewTilesArgs& p, int m) {
    C = p.C; W = p.W; H = p.H; KW = p.KW; K = p.K; dh = p.dh; dw = p.dw;
    magic_c = p.magic_c; magic_kw = p.magic_kw;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.data), 0,
                                             static_cast<uint32_t>(p.images) * p.H * p.W * p.C,
                                             0x00020000);
    ok = m < p.M;
    const int mm = ok ? m : 0, plane = p.OH * p.OW;
    const int n = mm / plane, rem = mm - n * plane;
    const int oh = rem / p.OW, ow = rem - oh * p.OW;
    ih0 = oh * p.sh - p.ph;
    iw0 = ow * p.sw - p.pw;
    pix = ((n * H + ih0) * W + iw0) * C;
  }
  __device__ __forceinline__ v4i load(int k0) const {
    const int tap = few_tiles_div(k0 >> 4, magic_c), c = k0 - tap * C;
    const int kh = few_tiles_div(tap, magic_kw), kw = tap - kh * KW;
    const int dih = kh * dh, diw = kw * dw;
    const bool in = ok && k0 < K && static_cast<unsigned>(ih0 + dih) < static_cast<unsigned>(H) &&
                    static_cast<unsigned>(iw0 + diw) < static_cast<unsigned>(W);
    const uint32_t off = in ? static_cast<uint32_t>(pix + (dih * W + diw) * C + c) : kOutOfRange;
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
  }
};

enum Operands { kAligned, kAny, kConv };

// T: rows and columns of an output tile, 32 or 16
template <int W, int T, int OPERANDS, int MODE>
__device__ __forceinline__ void few_tiles(const FewTilesArgs& p, int block) {
  constexpr int kDepth = depth_of(W, T), kTile = T, F = T / 16;
  constexpr int kPitch = T + 4;  // ints per row of a partial tile in LDS
  __shared__ __attribute__((aligned(16))) int part[W][kTile * kPitch];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = (p.N + kTile - 1) / kTile;
  const int tm = block / tiles_n, tn = block - tm * tiles_n;
  const int m0 = tm * kTile, n0 = tn * kTile;
  // how a lane loads (row, 16-byte piece of the row's 64) and what it multiplies
  const int load_row = lane >> 2, load_piece = lane & 3;
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int from_lane = 4 * (lrow * 4 + lgrp);
  auto to_mfma = [&](v4i v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_ds_bpermute(from_lane, v[i]);
    return v;
  };

  typename std::conditional<OPERANDS == kAny, AnyRows, AlignedRows>::type b[F];
  typename std::conditional<
      OPERANDS == kAny, AnyRows,
      typename std::conditional<OPERANDS == kConv, ConvRows, AlignedRows>::type>::type a[F];
#pragma unroll
  for (int i = 0; i < F; ++i) {
    if constexpr (OPERANDS == kConv)
      a[i].init(p, m0 + 16 * i + load_row);
    else
      a[i].init(p.data, m0 + 16 * i + load_row, p.M, p.K);
    b[i].init(p.weight, n0 + 16 * i + load_row, p.N, p.K);
  }

  v4i fa[kDepth][kSteps][F], fb[kDepth][kSteps][F];
  auto fetch = [&](int block, v4i (&x)[kSteps][F], v4i (&y)[kSteps][F]) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int k0 = block * kBlockK + s * 64 + load_piece * 16;
#pragma unroll
      for (int i = 0; i < F; ++i) {
        x[s][i] = a[i].load(k0);
        y[s][i] = b[i].load(k0);
      }
    }
  };
  const int blocks = (p.K + kBlockK - 1) / kBlockK;
  const int rounds = (blocks + W - 1) / W;
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
    if (d < rounds) fetch(wave + d * W, fa[d], fb[d]);

  // what the epilogue needs, behind the first loads: thread t finishes columns 4 * (t % Q) ... of
  // row t / Q, Q = T / 4 (and of row t / Q + 64 * W / Q with few waves)
  constexpr int Q = T / 4, kQuads = T * Q, kThreads = 64 * W;
  constexpr int kPer = (kQuads + kThreads - 1) / kThreads;
  const EpiPreOf<MODE> pre = epi_prefetch_scalars<MODE>(p.epi);
  const int n = n0 + 4 * (tid % Q);
  int bias[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    bias[i] = (tid < kQuads && n + i < p.N) ? epi_bias32(p.epi, pre.s, n + i) : 0;

  uint32_t residual[kPer];
  if constexpr (epi_sums(MODE)) {
    const bool dwords = epi_quad_dwords<MODE>(p.epi, p.N, static_cast<size_t>(p.ldo));
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int q = tid + j * kThreads, m = m0 + q / Q;
      residual[j] = 0;
      if (dwords && q < kQuads && m < p.M && n < p.N)
        residual[j] = *reinterpret_cast<const uint32_t*>(p.epi.res +
                                                         static_cast<size_t>(m) * p.ldo + n);
    }
  }

  // lane: activation row lane % 16, output columns 4 * (lane / 16) ... + 3
  v4i acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = v4i{0, 0, 0, 0};
  for (int r = 0; r < rounds; r += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      if (r + d < rounds) {
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          v4i x[F], y[F];
#pragma unroll
          for (int i = 0; i < F; ++i) {
            x[i] = to_mfma(fa[d][s][i]);
            y[i] = to_mfma(fb[d][s][i]);
          }
#pragma unroll
          for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
              acc[i][j] =
                  __builtin_amdgcn_mfma_i32_16x16x64_i8(y[j], x[i], acc[i][j], 0, 0, 0);
        }
        if (r + d + kDepth < rounds) fetch(wave + (r + d + kDepth) * W, fa[d], fb[d]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
      *reinterpret_cast<v4i*>(&part[wave][(16 * i + lrow) * kPitch + 16 * j + 4 * lgrp]) =
          acc[i][j];
  __syncthreads();

  if (block == 0 && tid == 0) epilogue_ranges<MODE>(p.epi);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int q = tid + j * kThreads;
    if (kQuads % kThreads != 0 && q >= kQuads) break;
    const int row = q / Q, m = m0 + row;
    uint32_t sum[4] = {};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const v4i x = *reinterpret_cast<const v4i*>(&part[w][row * kPitch + 4 * (tid % Q)]);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += static_cast<uint32_t>(x[i]);
    }
    if (m >= p.M || n >= p.N) continue;
    int v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = static_cast<int>(sum[i] + static_cast<uint32_t>(bias[i]));
    epi_store_quad<MODE>(p.epi, pre, v, m, n, p.N, static_cast<size_t>(p.ldo),
                         epi_sums(MODE) ? residual[j] : 0);
  }
}

template <int W, int T, int OPERANDS, int MODE>
__global__ __launch_bounds__(64 * W) void few_tiles_kernel(FewTilesArgs p) {
  few_tiles<W, T, OPERANDS, MODE>(p, blockIdx.x);
}

// Two convolutions of the same images in one launch.
struct FewTilesPair {
  FewTilesArgs a, b;
  int first;  // work-groups of a
};
template <int W, int T>
__global__ __launch_bounds__(64 * W) void few_tiles_pair_kernel(FewTilesPair p) {
  const bool second = static_cast<int>(blockIdx.x) >= p.first;
  FewTilesArgs a = p.a;
  if (second) a = p.b;
  few_tiles<W, T, kConv, kEpiPlain>(a, static_cast<int>(blockIdx.x) - (second ? p.first : 0));
}

// Rows of K bytes -> rows of Kp >= K bytes on 16-byte marks, zeros behind: two tensors in one
// launch, one 16-byte piece per lane.
struct PadJob {
  const int8_t* in;
  v4i* out;
  int rows;
  size_t pieces;
};
__global__ __launch_bounds__(256) void pad_rows_kernel(PadJob x, PadJob y, int K, int per_row) {
  size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
  const bool second = i >= x.pieces;
  if (second) i -= x.pieces;
  const int8_t* in = second ? y.in : x.in;
  v4i* out = second ? y.out : x.out;
  const bool ok = i < (second ? y.pieces : x.pieces);
  const size_t row = i / per_row;
  AnyRows r;
  r.base = in;
  r.K = K;
  r.total = static_cast<long long>(second ? y.rows : x.rows) * K;
  r.ok = ok;
  r.row = ok ? static_cast<long long>(row) * K : 0;
  const v4i v = r.load(static_cast<int>(i - row * per_row) * 16);
  if (ok) out[i] = v;
}

template <int OPERANDS, int MODE>
void launch(hipStream_t s, const FewTilesArgs& a, int waves) {
  const long side = waves == -4 || waves == -8 ? 16 : 32;
  const dim3 grid(static_cast<unsigned>((a.M + side - 1) / side * ((a.N + side - 1) / side)));
  switch (waves) {
    case -4:
      hipLaunchKernelGGL((few_tiles_kernel<4, 16, OPERANDS, MODE>), grid, dim3(256), 0, s, a);
      break;
    case -8:
      hipLaunchKernelGGL((few_tiles_kernel<8, 16, OPERANDS, MODE>), grid, dim3(512), 0, s, a);
      break;
    case 2:
      hipLaunchKernelGGL((few_tiles_kernel<2, 32, OPERANDS, MODE>), grid, dim3(128), 0, s, a);
      break;
    case 4:
      hipLaunchKernelGGL((few_tiles_kernel<4, 32, OPERANDS, MODE>), grid, dim3(256), 0, s, a);
      break;
    case 8:
      hipLaunchKernelGGL((few_tiles_kernel<8, 32, OPERANDS, MODE>), grid, dim3(512), 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((few_tiles_kernel<16, 32, OPERANDS, MODE>), grid, dim3(1024), 0, s, a);
  }
  MXQ_LAUNCH_CHECK();
}

template <int MODE>
void launch_rows(hipStream_t s, const FewTilesArgs& a, bool aligned, int waves) {
  if (aligned)
    launch<kAligned, MODE>(s, a, waves);
  else
    launch<kAny, MODE>(s, a, waves);
}

}  // namespace

// 16 x 16 tiles (negative) where 32 x 32 ones would occupy half of the CUs or fewer: a CU then takes
// in half the bytes and four times as many of them do (3 x 3 over 512 channels of one 7 x 7 plane
// 8.5 us -> 5.4, over 256 channels of 14 x 14 6.9 -> 4.5, 64 x 2048 -> 1000 5.0 -> 3.75; an empty
// launch is 3.0).  Between half and all of them the narrow tiles read too much twice (784 x 512 ->
// 256 5.0 us against 3.9).  There a wave per block of the reduction up to 8, up to 16 where the
// pieces are masked on their way in or the reduction has 16 blocks, which is level at worst.  With more tiles than the chip has CUs the
// tiles themselves fill it and splitting a reduction further only adds partial tiles (1024 x 435 ->
// 1024: 7.7 us on 2 waves, 14.3 on 8).
int few_tiles_waves(int M, int N, int K, bool aligned) {
  const int blocks = (K + kBlockK - 1) / kBlockK;
  const long tiles = few_tiles_count(M, N), cus = num_cus();
  if (2 * tiles <= cus && blocks > 1) return K >= 512 ? -8 : -4;
  if (tiles > 2 * cus || blocks <= 2) return 2;
  if (tiles > cus || blocks <= 4) return 4;
  return blocks > (aligned ? 15 : 8) ? 16 : 8;
}

void launch_few_tiles_fc(hipStream_t s, const FewTilesArgs& a, bool aligned, int waves) {
  MXQ_CHECK(static_cast<long long>(a.M) * a.K >= 16 && static_cast<long long>(a.N) * a.K >= 16,
            "operands below 16 bytes");
  switch (epi_mode(a.epi)) {
    case kEpiF32: launch_rows<kEpiF32>(s, a, aligned, waves); break;
    case kEpiSum: launch_rows<kEpiSum>(s, a, aligned, waves); break;
    case kEpiSumRq: launch_rows<kEpiSumRq>(s, a, aligned, waves); break;
    default: launch_rows<kEpiPlain>(s, a, aligned, waves);
  }
}

void launch_pad_rows(hipStream_t s, const int8_t* x, long long x_rows, int8_t* x_out,
                     const int8_t* y, long long y_rows, int8_t* y_out, int K, int Kp) {
  MXQ_CHECK(x_rows * K >= 16 && y_rows * K >= 16, "operands below 16 bytes");
  MXQ_CHECK(x_rows < (1LL << 31) && y_rows < (1LL << 31) && Kp % 16 == 0 && Kp >= K, "bad rows");
  const int per_row = Kp / 16;
  PadJob a = {x, reinterpret_cast<v4i*>(x_out), static_cast<int>(x_rows),
              static_cast<size_t>(x_rows) * per_row};
  PadJob b = {y, reinterpret_cast<v4i*>(y_out), static_cast<int>(y_rows),
              static_cast<size_t>(y_rows) * per_row};
  const size_t grid = (a.pieces + b.pieces + 255) / 256;
  MXQ_CHECK(grid < (size_t(1) << 31), "operands too large for one launch");
  hipLaunchKernelGGL(pad_rows_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, a, b, K,
                     per_row);
  MXQ_LAUNCH_CHECK();
}

bool few_tiles_conv_ok(int C, int K, int KH, int KW) {
  return C % 16 == 0 && static_cast<long long>(K / 16) * (C / 16) < (1LL << 32) &&
         static_cast<long long>(KH) * KW * KW < (1LL << 32);
}

static void conv_magics(FewTilesArgs& a) {
  auto magic = [](int d) {
    return d == 1 ? 0u : static_cast<uint32_t>((1ULL << 32) / static_cast<unsigned>(d) + 1);
  };
  a.magic_c = magic(a.C / 16);
  a.magic_kw = magic(a.KW);
}

void launch_few_tiles_conv(hipStream_t s, FewTilesArgs a, int waves) {
  conv_magics(a);
  launch<kConv, kEpiPlain>(s, a, waves);
}

void launch_few_tiles_pair(hipStream_t s, const FewTilesArgs& a, const FewTilesArgs& b, int waves) {
  FewTilesPair p = {a, b, 0};
  conv_magics(p.a);
  conv_magics(p.b);
  const long side = waves == -4 || waves == -8 ? 16 : 32;
  auto tiles = [&](const FewTilesArgs& x) {
    return static_cast<int>((x.M + side - 1) / side * ((x.N + side - 1) / side));
  };
  p.first = tiles(a);
  const dim3 grid(static_cast<unsigned>(p.first + tiles(b)));
  switch (waves) {
    case -4: hipLaunchKernelGGL((few_tiles_pair_kernel<4, 16>), grid, dim3(256), 0, s, p); break;
    case -8: hipLaunchKernelGGL((few_tiles_pair_kernel<8, 16>), grid, dim3(512), 0, s, p); break;
    case 2: hipLaunchKernelGGL((few_tiles_pair_kernel<2, 32>), grid, dim3(128), 0, s, p); break;
    case 4: hipLaunchKernelGGL((few_tiles_pair_kernel<4, 32>), grid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL((few_tiles_pair_kernel<8, 32>), grid, dim3(512), 0, s, p);
  }
  MXQ_LAUNCH_CHECK();
}

}  // namespace mxq
