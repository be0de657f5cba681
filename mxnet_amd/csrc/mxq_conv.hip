// _contrib_quantized_conv on gfx950: implicit-GEMM int8 convolution on NHWC
// operands with the same MFMA core and epilogue as the fully-connected kernel.
// Replaces cudnnConvolutionForward (NHWC int8, IMPLICIT_PRECOMP_GEMM), the
// float->int32 cast and QuantizedBiasAddKernel of the reference's GPU operator
// (src/operator/quantization/quantized_conv.cu:101-219); the accumulator stays an
// exact int32 and the bias is added in integers.
//
// GEMM view: rows m = (n, oh, ow), columns = output channel o, reduction
// k = (kh, kw, c) with c fastest, which is the memory order of both the NHWC
// activation pixel and the OHWI weight row.  Out-of-image taps and the K tail are
// zero-filled by the loader, so no padded copy of the input is ever made.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_few_tiles.h"
#include "mxq_resident.h"
#include "mxq_thin_transpose.h"
#include "mxq_gemm.h"
#include "mxq_tiles.h"

namespace mxq {

void launch_fc(hipStream_t s, const int8_t* data, const int8_t* weight, int M, int N, int K,
               int ldo, const Epilogue& epi, const GemmForce& force, const Workspace& ws);
size_t fc_workspace_bytes(int M, int N, int K, bool fused8);

namespace {

struct ConvArgs {
  const int8_t* data;    // [N][H][W][C]
  const int8_t* weight;  // [O][KH][KW][C]
  int N, H, W, C, O, KH, KW;
  int sh, sw, ph, pw, dh, dw, OH, OW;
  int M, K;  // N*OH*OW, KH*KW*C
  Epilogue epi;
  SplitK sk;
};

// Activation loader: row = output pixel, chunk = 16 channels of one filter tap.
template <class Cfg, int CHUNKS, bool ALIGNED>
struct ConvFetch {
  const int8_t* img[CHUNKS];  // start of image n
  int ih0[CHUNKS], iw0[CHUNKS];
  bool ok[CHUNKS];
  int lc;
  int C, KW, H, W, K, dh, dw;

  __device__ __forceinline__ void init(const ConvArgs& args, int row0) {
    C = args.C; KW = args.KW; H = args.H; W = args.W; K = args.K;
    dh = args.dh; dw = args.dw;
    lc = threadIdx.x % Cfg::CH;
    const int lr = threadIdx.x / Cfg::CH;
    const int ohow = args.OH * args.OW;
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
      const int m = row0 + lr + j * Cfg::ROWS_PER_PASS;
      ok[j] = m < args.M;
      const int mm = ok[j] ? m : 0;
      const int n = mm / ohow;
      const int rem = mm - n * ohow;
      const int oh = rem / args.OW;
      const int ow = rem - oh * args.OW;
      img[j] = args.data + static_cast<size_t>(n) * args.H * args.W * args.C;
      ih0[j] = oh * args.sh - args.ph;
      iw0[j] = ow * args.sw - args.pw;
    }
  }

  __device__ __forceinline__ void fetch(int kt, v4i (&reg)[CHUNKS]) {
    const int k0 = kt * Cfg::BK + lc * 16;
    if (ALIGNED) {
      // C % 16 == 0: the 16 bytes lie inside one tap
      const bool k_ok = k0 < K;
      const int tap = k0 / C;
      const int c = k0 - tap * C;
      const int kh = tap / KW;
      const int kw = tap - kh * KW;
      const int dih = kh * dh, diw = kw * dw;
#pragma unroll
      for (int j = 0; j < CHUNKS; ++j) {
        const int ih = ih0[j] + dih, iw = iw0[j] + diw;
        const bool v = ok[j] && k_ok && ih >= 0 && ih < H && iw >= 0 && iw < W;
        v4i r = {0, 0, 0, 0};
        if (v)
          r = *reinterpret_cast<const v4i*>(img[j] +
                                            (static_cast<size_t>(ih) * W + iw) * C + c);
        reg[j] = r;
      }
    } else {
#pragma unroll
      for (int j = 0; j < CHUNKS; ++j) {
        v4i r = {0, 0, 0, 0};
        if (ok[j]) {
          for (int i = 0; i < 16; ++i) {
            const int k = k0 + i;
            if (k >= K) break;
            const int tap = k / C;
            const int c = k - tap * C;
            const int kh = tap / KW;
            const int kw = tap - kh * KW;
            const int ih = ih0[j] + kh * dh, iw = iw0[j] + kw * dw;
            if (ih >= 0 && ih < H && iw >= 0 && iw < W) {
              uint32_t b =
                  static_cast<uint8_t>(img[j][(static_cast<size_t>(ih) * W + iw) * C + c]);
              r[i >> 2] |= static_cast<int>(b << (8 * (i & 3)));
            }
          }
        }
        reg[j] = r;
      }
    }
  }
};

template <class Cfg, bool ALIGNED>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kMinWaves) void conv_kernel(ConvArgs p) {
  __shared__ __attribute__((aligned(16))) v4i lds[2][Cfg::STAGE_SLOTS];
  const int wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.O + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;

  ConvFetch<Cfg, Cfg::A_CHUNKS, ALIGNED> af;
  RowFetch<Cfg, Cfg::B_CHUNKS, ALIGNED> bf;
  af.init(p, m0);
  bf.init(p.weight, n0, p.O, p.K);

  v16i acc[Cfg::MI][Cfg::NI];
  gemm_mainloop<Cfg>(acc, af, bf, (p.K + Cfg::BK - 1) / Cfg::BK, lds);

  gemm_epilogue<Cfg>(acc, p.epi, m0 + wm * Cfg::TM, n0 + wn * Cfg::TN, p.M, p.O,
                     static_cast<size_t>(p.O));
  if (blockIdx.x == 0 && threadIdx.x == 0) epilogue_ranges(p.epi);
}

// Activation operand of the direct-to-LDS main loop: lane state for "16 channels of
// one filter tap of one output pixel", advanced stage by stage without divisions.
// Halo taps, rows past the last pixel and the K tail are sent to an out-of-range
// buffer offset and arrive in LDS as zeros.  Needs C % 16 == 0.
template <class Cfg, int INSTR>
struct ConvIssuer {
  int pix[INSTR];           // byte offset of pixel (n, ih0, iw0), may be negative
  int ih0[INSTR], iw0[INSTR];
  bool ok[INSTR];
  int cc, kh, kw;           // position of this lane's chunk in the stage issued next
  int dih, diw, tapoff;     // kh*dilate_h, kw*dilate_w, ((kh*dh)*W + kw*dw)*C
  int C, H, W, KH, KW, dh, dw;
  v4i rsrc;

  // kbeg: reduction index (a multiple of the stage depth) at which stage 0 starts
  __device__ __forceinline__ void init(const ConvArgs& a, int row_begin, int wave, int lane,
                                       int kbeg = 0) {
    C = a.C; H = a.H; W = a.W; KH = a.KH; KW = a.KW; dh = a.dh; dw = a.dw;
    rsrc = make_rsrc(a.data, static_cast<uint32_t>(a.N) * a.H * a.W * a.C);
    DmaLane<Cfg> g;
    g.init(wave, lane);
    const int k = kbeg + g.c16;
    const int tap = k / C;
    cc = k - tap * C;
    kh = tap / KW;
    kw = tap - kh * KW;
    retap();
    const int ohow = a.OH * a.OW;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int m = row_begin + g.row0 + i * DmaLane<Cfg>::kRowStep;
      ok[i] = m < a.M;
      const int mm = ok[i] ? m : 0;
      const int n = mm / ohow;
      const int rem = mm - n * ohow;
      const int oh = rem / a.OW;
      const int ow = rem - oh * a.OW;
      ih0[i] = oh * a.sh - a.ph;
      iw0[i] = ow * a.sw - a.pw;
      pix[i] = ((n * H + ih0[i]) * W + iw0[i]) * C;
    }
  }
  __device__ __forceinline__ void retap() {
    dih = kh * dh;
    diw = kw * dw;
    tapoff = (dih * W + diw) * C;
  }
  __device__ __forceinline__ void issue(int i, int, uint32_t lds_addr) {
    const int ih = ih0[i] + dih, iw = iw0[i] + diw;
    const bool v = ok[i] && kh < KH && static_cast<unsigned>(ih) < static_cast<unsigned>(H) &&
                   static_cast<unsigned>(iw) < static_cast<unsigned>(W);
    const uint32_t off = v ? static_cast<uint32_t>(pix[i] + tapoff + cc) : kOutOfRange;
    dma_buffer(lds_addr, off, rsrc);
  }
  __device__ __forceinline__ void stage_done() {
    cc += Cfg::BK;
    while (cc >= C) {
      cc -= C;
      if (++kw == KW) {
        kw = 0;
        ++kh;
      }
    }
    retap();
  }
};

template <class Cfg, int NS, int PIPE>
__device__ __forceinline__ void conv_dma(const ConvArgs& p, int block) {
  __shared__ __attribute__((aligned(16))) v4i lds[NS * Cfg::STAGE_SLOTS];
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.O + Cfg::BN - 1) / Cfg::BN;
  int tm, tn, tile = 0, z = 0;
  if (__builtin_expect(p.sk.splits > 1, 0))
    tile_coords_split(block, tiles_m, tiles_n, p.sk.splits, tm, tn, tile, z);
  else
    tile_coords(block, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // what the epilogue needs is fetched while the first operand stages are in flight
  EpiPreOf<kEpiPlain> pre;
  auto prefetch = [&]() { pre = epi_prefetch<Cfg>(p.epi, n0, p.O); };
  // this work-group's K slice: stages [kt0, kt0 + KT) (all of them without a split)
  const int kt_all = (p.K + Cfg::BK - 1) / Cfg::BK;
  const int kt0 = z * p.sk.kt_per_split;
  const int KT = (kt_all - kt0) < p.sk.kt_per_split ? (kt_all - kt0) : p.sk.kt_per_split;
  const int kbeg = kt0 * Cfg::BK;
  ConvIssuer<Cfg, Cfg::A_CHUNKS> ai;
  RowIssuerBuffer<Cfg, Cfg::B_CHUNKS> bi;
  ai.init(p, m0, wave, lane, kbeg);
  bi.init(p.weight, n0, p.O, p.K, wave, lane, kbeg);

  v16i acc[Cfg::MI][Cfg::NI];
  gemm_mainloop_dma<Cfg, NS, PIPE>(acc, ai, bi, KT, lds, prefetch);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (block == 0 && threadIdx.x == 0) epilogue_ranges(p.epi);
  if (__builtin_expect(p.sk.splits > 1, 0) && !splitk_gather<Cfg>(acc, p.sk, tile, z)) return;

  gemm_epilogue_lds<Cfg, NS * Cfg::STAGE_SLOTS * 16>(acc, p.epi, pre, m0, n0, p.M, p.O,
                                                     static_cast<size_t>(p.O), lds);
}

template <class Cfg, int NS, int PIPE>
__global__ __launch_bounds__(Cfg::kThreads, NS <= 2 ? Cfg::kMinWaves : 1) void conv_dma_kernel(ConvArgs p) {
  conv_dma<Cfg, NS, PIPE>(p, blockIdx.x);
}

// Tiles on eight waves (gemm_mainloop_sliced).
template <class Cfg, int NS>
__device__ __forceinline__ void conv_sliced(const ConvArgs& p, int block) {
  typedef typename Cfg::Tile Tile;
  __shared__ __attribute__((aligned(16))) v4i lds[NS * Cfg::STAGE_SLOTS];
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.O + Cfg::BN - 1) / Cfg::BN;
  int tm, tn, tile = 0, z = 0;
  if (__builtin_expect(p.sk.splits > 1, 0))
    tile_coords_split(block, tiles_m, tiles_n, p.sk.splits, tm, tn, tile, z);
  else
    tile_coords(block, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  EpiPreOf<kEpiPlain> pre;
  auto prefetch = [&]() { pre = epi_prefetch<Tile>(p.epi, n0, p.O); };
  const int kt_all = (p.K + Cfg::BK - 1) / Cfg::BK;
  const int kt0 = z * p.sk.kt_per_split;
  const int KT = (kt_all - kt0) < p.sk.kt_per_split ? (kt_all - kt0) : p.sk.kt_per_split;
  ConvIssuer<Cfg, Cfg::A_CHUNKS> ai;
  RowIssuerBuffer<Cfg, Cfg::B_CHUNKS> bi;
  ai.init(p, m0, wave, lane, kt0 * Cfg::BK);
  bi.init(p.weight, n0, p.O, p.K, wave, lane, kt0 * Cfg::BK);
  if (block == 0 && threadIdx.x == 0) epilogue_ranges(p.epi);
  v16i acc[1][Cfg::NI];
  if (!gemm_mainloop_sliced<Cfg, NS>(acc, ai, bi, KT, lds, prefetch)) return;
  if (__builtin_expect(p.sk.splits > 1, 0) && !splitk_gather<Tile>(acc, p.sk, tile, z)) return;
  gemm_epilogue_lds<Tile, NS * Cfg::STAGE_SLOTS * 16>(acc, p.epi, pre, m0, n0, p.M, p.O,
                                                      static_cast<size_t>(p.O), lds);
}

template <class Cfg, int NS>
__global__ __launch_bounds__(Cfg::kThreads, 2) void conv_sliced_kernel(ConvArgs p) {
  conv_sliced<Cfg, NS>(p, blockIdx.x);
}

// Two convolutions of the same images in one launch.
struct ConvPair {
  ConvArgs a, b;
  int first;  // work-groups of a
};
template <class Cfg, int NS>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kMinWaves) void conv_pair_kernel(ConvPair p) {
  const bool second = static_cast<int>(blockIdx.x) >= p.first;
  ConvArgs a = p.a;
  if (second) a = p.b;
  conv_dma<Cfg, NS, 0>(a, static_cast<int>(blockIdx.x) - (second ? p.first : 0));
}

// ---- 3 x 3 convolution over 64 channels with the weights parked in LDS --------------
// A layer like ResNet's 56 x 56, 64 -> 64 has a short reduction (K = 576) and a weight
// tensor of 36 KB: as an implicit GEMM every tile is prologue and epilogue, and the nine
// taps re-fetch every input pixel nine times.  Here a work-group of 8 waves parks the whole
// weight tensor in LDS once; after that one barrier every wave works on its own.  An item
// is R consecutive output rows of one image: the wave brings their R + 2 input rows (with
// the zero halo left and right, zero rows above and below the image) into its private LDS
// patch with buffer loads ... lds, then for each output row runs the 9 taps x 2 k-steps x
// (2 x 2) MFMAs out of LDS, adds the bias, requantizes and stores the row; the int8 tile is
// transposed through the patch row that has just become dead.  No barrier per K step,
// every input row is fetched (R + 2) / R times instead of nine, and with two waves per SIMD
// one wave's fetch and epilogue overlap the other's MFMAs.  int8 output with the fused
// requantize (the form the quantized graph runs with a calibrated convolution), or the operator's
// int32 planes: a register holds 32 consecutive pixels of one channel then, which leave as they
// are, 128 bytes a channel (56 x 56 at batch 64 26.6 -> 21.1 us, the tiled kernel before).
// Other outputs take the tiled kernels.
constexpr int kRowsC = 64;        // input channels = bytes per pixel
constexpr int kRowsO = 64;        // output channels
constexpr int kRowsPitch = 60;    // patch pixels per row
constexpr int kRowsMaxW = kRowsPitch - 2;
constexpr int kRowsWaves = 8;

// (row & 3) ^ (row >> 2 & 3): spreads the 16-byte pieces of the transposed int8 tile (row
// pitch 64 bytes) over the banks for the column-wise writes and the row-wise reads alike
__device__ __forceinline__ int tile_swz(int row) { return (row ^ (row >> 2)) & 3; }

// PLANES: int32 planes instead of int8 pixels
template <int R, bool PLANES>
__global__ __launch_bounds__(64 * kRowsWaves, 1) void conv3x3_rows_kernel(ConvArgs p) {
  constexpr int CH = kRowsC / 16;                       // 16-byte chunks per pixel
  constexpr int kPatchPixels = (R + 2) * kRowsPitch;
  constexpr int kFetches = (kPatchPixels + 15) / 16;    // buffer loads of 16 pixels each
  __shared__ __attribute__((aligned(16))) v4i wl[9 * kRowsO * CH];               // 36 KB
  __shared__ __attribute__((aligned(16))) v4i patch_all[kRowsWaves * kPatchPixels * CH];
  __shared__ __attribute__((aligned(16))) int sbias[kRowsO];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  v4i* patch = patch_all + wave * kPatchPixels * CH;
  const uint32_t patch_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(patch));
  const v4i rsrc = make_rsrc(p.data, static_cast<uint32_t>(p.N) * p.H * p.W * kRowsC);
  const int chunks_per_image = (p.OH + R - 1) / R;
  const int items = p.N * chunks_per_image;
  // lane geometry of the fetches: flat patch pixel 16 * j + lane / 4, chunk slot lane % 4
  auto fetch = [&](int item) {
    const int n = item / chunks_per_image, oh0 = (item - n * chunks_per_image) * R;
#pragma unroll
    for (int j = 0; j < kFetches; ++j) {
      const int flat = 16 * j + (lane >> 2);
      const int row = flat / kRowsPitch, px = flat - row * kRowsPitch;
      const int ih = oh0 + row - 1, iw = px - 1;
      const int chunk = (lane & 3) ^ swz<CH>(px);
      const bool ok = static_cast<unsigned>(ih) < static_cast<unsigned>(p.H) &&
                      static_cast<unsigned>(iw) < static_cast<unsigned>(p.W);
      const uint32_t off =
          ok ? static_cast<uint32_t>(((n * p.H + ih) * p.W + iw) * kRowsC + chunk * 16)
             : kOutOfRange;
      if (flat < kPatchPixels) dma_buffer(patch_addr + j * 1024, off, rsrc);
    }
  };
  int item = blockIdx.x * kRowsWaves + wave;
  if (item < items) fetch(item);  // on its way while the weights are staged

  // weights [o][tap][c] -> LDS [tap][o][chunk ^ swz(o)], straight into LDS as well: fetch
  // j fills the 16 rows (tap, o) = 16 * j ... + 15, lane / 4 the row, lane % 4 the slot
  {
    const v4i wrsrc = make_rsrc(p.weight, 9 * kRowsO * kRowsC);
    const uint32_t wl_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(wl));
    constexpr int kWeightFetches = 9 * kRowsO / 16;  // 36
    for (int j = wave; j < kWeightFetches; j += kRowsWaves) {
      const int row = 16 * j + (lane >> 2);
      const int t = row / kRowsO, o = row - t * kRowsO;
      const int chunk = (lane & 3) ^ swz<CH>(o);
      dma_buffer(wl_addr + j * 1024, static_cast<uint32_t>((o * 9 + t) * kRowsC + chunk * 16),
                 wrsrc);
    }
  }
  const EpiScalars s = epi_scalars(p.epi);
  if (tid < kRowsO) sbias[tid] = epi_bias32(p.epi, s, tid);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int lrow = lane & 31, lgrp = lane >> 5;
  const bool relu = p.epi.relu != 0, stream8 = p.epi.stream8 != 0;
  // patch pixel of output column mi * 32 + lrow under tap column kw; columns past the row
  // (their results are never stored) are kept inside it
  int apx[2][3];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int kw = 0; kw < 3; ++kw) {
      const int px = mi * 32 + lrow + kw;
      apx[mi][kw] = px < kRowsPitch ? px : kRowsPitch - 1;
    }
  for (; item < items; item += gridDim.x * kRowsWaves) {
    const int n = item / chunks_per_image, oh0 = (item - n * chunks_per_image) * R;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    // a real loop: the second row re-runs the first row's instructions out of the
    // instruction cache instead of fetching a second copy of them
#pragma unroll 1
    for (int r = 0; r < R; ++r) {
      if (oh0 + r >= p.OH) break;
      // accumulators start at the int32 bias of their columns, read from LDS straight into
      // the registers the MFMAs add to: no bias add in the epilogue
      v16i acc[2][2];
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const v4i b = *reinterpret_cast<const v4i*>(sbias + ni * 32 + 8 * vq + 4 * lgrp);
#pragma unroll
          for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[mi][ni][4 * vq + i] = b[i];
        }
#pragma unroll
      for (int kh = 0; kh < 3; ++kh)
#pragma unroll
        for (int kw = 0; kw < 3; ++kw)
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            v4i fa[2], fb[2];
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
              const int px = apx[mi][kw];
              fa[mi] = patch[((r + kh) * kRowsPitch + px) * CH + ((ks * 2 + lgrp) ^ swz<CH>(px))];
            }
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
              fb[ni] = wl[((kh * 3 + kw) * kRowsO + ni * 32 + lrow) * CH +
                          ((ks * 2 + lgrp) ^ swz<CH>(lrow))];
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
#pragma unroll
              for (int ni = 0; ni < 2; ++ni)
                acc[mi][ni] =
                    __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ni], fa[mi], acc[mi][ni], 0, 0, 0);
          }
      if constexpr (PLANES) {
        // (the products' wait states stand here: none behind the masks of the stores)
        asm volatile("s_nop 15\n\ts_nop 15"
                     : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[1][0]), "+v"(acc[1][1]));
        const int plane = p.OH * p.OW;
        const auto image = __builtin_amdgcn_make_buffer_rsrc(
            p.epi.out32 + static_cast<size_t>(n) * kRowsO * plane, 0, kRowsO * plane * 4,
            0x00020000);
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const int px = mi * 32 + lrow;
          // past the end of the row: dropped
          const uint32_t at = px < p.OW ? ((oh0 + r) * p.OW + px + 4 * lgrp * plane) * 4u
                                        : kOutOfRange;
#pragma unroll
          for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int v = 0; v < 16; ++v)
              __builtin_amdgcn_raw_buffer_store_b32(
                  static_cast<uint32_t>(acc[mi][ni][v]), image, at,
                  (ni * 32 + 8 * (v / 4) + v % 4) * plane * 4, 0);
        }
        continue;
      }
      // patch row r is dead now (output row r + 1 starts at patch row r + 1): the int8 tile
      // of up to 58 pixels x 64 channels is transposed through it, 64 bytes per pixel
      char* stage = reinterpret_cast<char*>(patch + r * kRowsPitch * CH);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
      auto requantize_tile = [&](auto with_relu) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const int px = mi * 32 + lrow;
#pragma unroll
          for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) {
              const int nl = ni * 32 + 8 * vq + 4 * lgrp;
              const uint32_t w = epi_requant_pack<decltype(with_relu)::value>(
                  acc[mi][ni][4 * vq], acc[mi][ni][4 * vq + 1], acc[mi][ni][4 * vq + 2],
                  acc[mi][ni][4 * vq + 3], s);
              if (px < p.OW)
                *reinterpret_cast<uint32_t*>(stage + px * kRowsO +
                                             (((nl >> 4) ^ tile_swz(px)) << 4) + (nl & 15)) = w;
            }
        }
      };
      if (relu)
        requantize_tile(std::true_type());
      else
        requantize_tile(std::false_type());
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
      int8_t* orow = p.epi.out8 +
                     (static_cast<size_t>(n) * p.OH + oh0 + r) * p.OW * kRowsO;
      auto store_row = [&](auto stream) {
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const int px = it * 16 + (lane >> 2), c16 = lane & 3;
          if (px < p.OW) {
            const v4i val =
                *reinterpret_cast<const v4i*>(stage + px * kRowsO + ((c16 ^ tile_swz(px)) << 4));
            epi_store16<decltype(stream)::value>(val, orow + px * kRowsO + c16 * 16);
          }
        }
      };
      if (stream8)
        store_row(std::true_type());
      else
        store_row(std::false_type());
    }
    // the next item's fetches overwrite the patch: every LDS read above must have returned
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int next = item + gridDim.x * kRowsWaves;
    if (next < items) fetch(next);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) epilogue_ranges(p.epi);
}

bool conv3x3_rows_ok(const ConvArgs& a) {
  const long long data_bytes = static_cast<long long>(a.N) * a.H * a.W * a.C;
  return a.KH == 3 && a.KW == 3 && a.sh == 1 && a.sw == 1 && a.ph == 1 && a.pw == 1 &&
         a.dh == 1 && a.dw == 1 && a.C == kRowsC && a.O == kRowsO && a.W <= kRowsMaxW &&
         aligned16(a.data) && aligned16(a.weight) && data_bytes < (1LL << 31) &&
         (a.epi.out32 == nullptr
              ? a.epi.out8 != nullptr && aligned16(a.epi.out8)
              : a.epi.out8 == nullptr && a.epi.plane > 0 &&
                    4LL * kRowsO * a.OH * a.OW < (1LL << 31));
}

struct RowItems {
  bool two;      // output rows per item, or one
  long items;
  long rounds;   // of the chip's waves over them
};
RowItems row_items(const ConvArgs& a) {
  const long waves = static_cast<long>(kRowsWaves) * num_cus();
  // two output rows per item once that still gives most waves of the chip an item: a third
  // fewer input rows to fetch per output row
  const long items2 = static_cast<long>(a.N) * ((a.OH + 1) / 2);
  RowItems r;
  r.two = 5 * items2 >= 3 * waves;
  r.items = r.two ? items2 : static_cast<long>(a.N) * a.OH;
  r.rounds = (r.items + waves - 1) / waves;
  return r;
}

void launch_conv3x3_rows(hipStream_t s, const ConvArgs& a) {
  const long cus = num_cus();
  const RowItems r = row_items(a);
  long grid = (r.items + kRowsWaves - 1) / kRowsWaves;
  if (grid > cus) grid = cus;
  const bool two = r.two;
  const auto kernel = a.epi.out32 != nullptr
                          ? (two ? conv3x3_rows_kernel<2, true> : conv3x3_rows_kernel<1, true>)
                          : (two ? conv3x3_rows_kernel<2, false> : conv3x3_rows_kernel<1, false>);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * kRowsWaves), 0, s, a);
  MXQ_LAUNCH_CHECK();
}

// Whether int32 planes leave this kernel sooner than the tiled one, which moves the wider output
// through LDS: from three rows a CU on (us, tiled and here, 56 x 56: 448 rows 7.6 / 8.4, 896 11.4 /
// 9.3, 1344 13.4 / 10.4, 3584 26.6 / 21.1), but not for short rows, whose products are mostly padding
// (28 wide, 1792 rows 11.3 / 9.7, 17 wide, 2624 rows 10.0 / 12.5, 14 wide, 3584 rows 11.0 / 13.1), nor
// for rows of less than 36 pixels where the last of several rounds leaves most waves idle (24 and
// 28 wide, 4600 rows: 12 and 9 % behind, 29 wide 4484 rows 28.1 / 31.6; 9000 rows 2 % behind and
// 3 % ahead), and less than five a CU (32 wide, 800 rows 11.8 / 12.9).
bool conv3x3_rows_wins_planes(const ConvArgs& a) {
  const long rows = static_cast<long>(a.N) * a.OH;
  if (a.W < 24 || rows < (a.W >= 36 ? 3L : 5L) * num_cus()) return false;
  const RowItems r = row_items(a);
  const long room = r.rounds * kRowsWaves * num_cus();
  return a.W >= 36 || r.rounds == 1 || 10 * room <= 16 * r.items;
}

// ---- few-tap convolution over 16 channels, straight from memory -------------------------
// An image's first layer (16 channels, usually 12 real ones in space-to-depth form) has a
// reduction of one 16-byte piece per tap: 256 bytes for a 7 x 7 stride-2 stem.  As tiles of the
// implicit GEMM that is 12544 work-groups of four stages, each with its own prologue, im2col
// gather through LDS and epilogue (batch 64, 224 x 224: 57 us).  Consecutive output pixels of a
// row read consecutive 16-byte pixels, so the MFMA's activation fragment (32 pixels by two taps)
// is one coalesced load per lane and needs no LDS at all.  A work-group parks the weights in LDS
// once and walks a contiguous run of pixels, 32 at a time per wave, the next 32 pixels' fragments
// requested before the current ones are multiplied: 27 us, of which the matrix products, the
// requantization's arithmetic and the 64 MB of memory traffic need 11 to 12 each.
// int8 output with the fused requantize; `strips` groups of 32 * NI output channels.
struct TapArgs {
  ConvArgs c;
  int items_per_group;  // 32-pixel tiles times strips that one work-group walks
  int strips;
};

template <int KS, int NI>
__global__ __launch_bounds__(256, KS > 5 ? 3 : 4) void conv_taps_kernel(TapArgs t) {
  const ConvArgs& p = t.c;
  constexpr int TN = 32 * NI, LD = TN + 16, LPR = TN / 16, RPI = 64 / LPR;
  constexpr int CH = 2 * KS, PITCH = CH | 1;  // 16-byte pieces per weight row; odd against banks
  extern __shared__ __attribute__((aligned(16))) char taps_lds[];
  const int rows = t.strips * TN;
  v4i* wl = reinterpret_cast<v4i*>(taps_lds);                                   // [rows][PITCH]
  int* sbias = reinterpret_cast<int*>(wl + rows * PITCH);                       // [rows]
  char* stage_all = reinterpret_cast<char*>(sbias + rows);                      // [4][32 * LD]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lgrp = lane >> 5;
  const int taps = p.KH * p.KW;
  for (int i = tid; i < rows * CH; i += 256) {
    const int o = i / CH, c = i - o * CH;
    v4i w = {0, 0, 0, 0};
    if (o < p.O && c < taps)
      w = *reinterpret_cast<const v4i*>(p.weight + (static_cast<size_t>(o) * taps + c) * 16);
    wl[o * PITCH + c] = w;
  }
  const EpiScalars s = epi_scalars(p.epi);
  for (int i = tid; i < rows; i += 256) sbias[i] = i < p.O ? epi_bias32(p.epi, s, i) : 0;
  __syncthreads();

  // this lane's taps: 2 * ks + lane / 32 (taps past the last one meet zero weights; they re-read
  // the window's first pixel)
  int dih[KS], diw[KS], toff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int tap = 2 * ks + lgrp < taps ? 2 * ks + lgrp : 0;
    const int kh = tap / p.KW, kw = tap - kh * p.KW;
    dih[ks] = kh * p.dh;
    diw[ks] = kw * p.dw;
    toff[ks] = (dih[ks] * p.W + diw[ks]) * 16;
  }
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(p.data), 0, static_cast<uint32_t>(p.N) * p.H * p.W * 16, 0x00020000);
  const int reach_h = (p.KH - 1) * p.dh, reach_w = (p.KW - 1) * p.dw;
  const int tiles = (p.M + 31) / 32, items = tiles * t.strips;
  int item = blockIdx.x * t.items_per_group + wave;
  const int end = (blockIdx.x + 1) * t.items_per_group < items
                      ? (blockIdx.x + 1) * t.items_per_group : items;
  // the lane's output pixel, moved on from item to item without a division
  const int plane = p.OH * p.OW;
  int tile = item / t.strips, strip = item - tile * t.strips;
  int n, oh, ow;
  {
    const int m = tile * 32 + lrow;
    n = m / plane;
    const int rem = m - n * plane;
    oh = rem / p.OW;
    ow = rem - oh * p.OW;
  }
  auto advance = [&](int by) {  // by tiles
    if (by == 0) return;
    ow += by * 32;
    while (ow >= p.OW) {
      ow -= p.OW;
      if (++oh == p.OH) {
        oh = 0;
        ++n;
      }
    }
  };
  // `more` == false: nothing is fetched, but the loads are issued all the same (kOutOfRange): a
  // branch around them would make every turn of the loop wait for its own prefetch
  auto load_a = [&](v4i (&f)[KS], bool more) {
    const int ih0 = oh * p.sh - p.ph, iw0 = ow * p.sw - p.pw;
    const int base = ((n * p.H + ih0) * p.W + iw0) * 16;
    const bool live = more && n < p.N;
    const bool inside = live && ih0 >= 0 && iw0 >= 0 && ih0 + reach_h < p.H && iw0 + reach_w < p.W;
    if (__all(inside)) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        f[ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                            rsrc, static_cast<uint32_t>(base + toff[ks]), 0, 0));
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool ok = live &&
                        static_cast<unsigned>(ih0 + dih[ks]) < static_cast<unsigned>(p.H) &&
                        static_cast<unsigned>(iw0 + diw[ks]) < static_cast<unsigned>(p.W);
        f[ks] = __builtin_bit_cast(
            v4i, __builtin_amdgcn_raw_buffer_load_b128(
                     rsrc, ok ? static_cast<uint32_t>(base + toff[ks]) : kOutOfRange, 0, 0));
      }
    }
  };
  char* stage = stage_all + wave * 32 * LD;
  auto turn = [&](const v4i (&fa)[KS], v4i (&fa_next)[KS], auto with_relu, auto stream) {
    const int m_base = tile * 32, s0 = strip * TN;
    const bool more = item + 4 < end;
    if (more) {
      const int next = (item + 4) / t.strips;
      advance(next - tile);
      strip = item + 4 - next * t.strips;
      tile = next;
    }
    load_a(fa_next, more);
    v16i acc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const v4i b = *reinterpret_cast<const v4i*>(sbias + s0 + ni * 32 + 8 * vq + 4 * lgrp);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[ni][4 * vq + i] = b[i];
      }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
            wl[(s0 + ni * 32 + lrow) * PITCH + 2 * ks + lgrp], fa[ks], acc[ni], 0, 0, 0);
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq)
        *reinterpret_cast<uint32_t*>(stage + lrow * LD + ni * 32 + 8 * vq + 4 * lgrp) =
            epi_requant_pack<decltype(with_relu)::value>(acc[ni][4 * vq], acc[ni][4 * vq + 1],
                                                         acc[ni][4 * vq + 2],
                                                         acc[ni][4 * vq + 3], s);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    // rows past the last pixel lie past the descriptor's end and are dropped
    const int left = p.M - m_base < 32 ? p.M - m_base : 32;
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        p.epi.out8 + static_cast<size_t>(m_base) * p.O, 0, left * p.O, 0x00020000);
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it) {
      const int rr = it * RPI + lane / LPR, c16 = lane % LPR, o = s0 + c16 * 16;
      const v4i val = *reinterpret_cast<const v4i*>(stage + rr * LD + c16 * 16);
      __builtin_amdgcn_raw_buffer_store_b128(
          val, out, o < p.O ? static_cast<uint32_t>(rr * p.O + o) : kOutOfRange, 0,
          decltype(stream)::value ? 2 /* nt */ : kDeviceScope);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    item += 4;
  };
  // two sets of fragments change places instead of being copied: a copy would wait for its loads
  auto run = [&](auto with_relu, auto stream) {
    v4i x[KS], y[KS];
    load_a(x, item < end);
    while (item < end) {
      turn(x, y, with_relu, stream);
      if (item >= end) break;
      turn(y, x, with_relu, stream);
    }
  };
  if (p.epi.stream8) {
    if (p.epi.relu)
      run(std::true_type(), std::true_type());
    else
      run(std::false_type(), std::true_type());
  } else if (p.epi.relu) {
    run(std::true_type(), std::false_type());
  } else {
    run(std::false_type(), std::false_type());
  }
  if (blockIdx.x == 0 && tid == 0) epilogue_ranges(p.epi);
}

bool conv_taps_ok(const ConvArgs& a) {
  const long long data_bytes = static_cast<long long>(a.N) * a.H * a.W * a.C;
  return a.C == 16 && a.KH * a.KW <= 16 && a.KH * a.KW > 1 && a.O % 16 == 0 && a.O <= 128 &&
         a.epi.out32 == nullptr && a.epi.out8 != nullptr && aligned16(a.data) &&
         aligned16(a.weight) && aligned16(a.epi.out8) && data_bytes < (1LL << 31);
}

template <int KS, int NI>
void launch_taps(hipStream_t s, const ConvArgs& a) {
  TapArgs t;
  t.c = a;
  t.strips = (a.O + 32 * NI - 1) / (32 * NI);
  const int rows = t.strips * 32 * NI;
  const long items = static_cast<long>((a.M + 31) / 32) * t.strips;
  // as many work-groups as the CUs hold at once; runs of whole rounds of the four waves
  const long groups = (KS > 5 ? 3L : 4L) * num_cus();
  long per = ((items + groups - 1) / groups + 3) / 4 * 4;
  t.items_per_group = static_cast<int>(per);
  const size_t lds = static_cast<size_t>(rows) * ((2 * KS) | 1) * 16 + rows * 4 +
                     4 * 32 * (32 * NI + 16);
  hipLaunchKernelGGL((conv_taps_kernel<KS, NI>),
                     dim3(static_cast<unsigned>((items + per - 1) / per)), dim3(256), lds, s, t);
  MXQ_LAUNCH_CHECK();
}

void launch_conv_taps(hipStream_t s, const ConvArgs& a) {
  const int ks = (a.KH * a.KW + 1) / 2;
#define MXQ_TAPS(KS)                  \
  do {                                \
    if (a.O <= 32)                    \
      launch_taps<KS, 1>(s, a);       \
    else                              \
      launch_taps<KS, 2>(s, a);       \
  } while (0)
  if (ks <= 2) MXQ_TAPS(2); else if (ks <= 5) MXQ_TAPS(5); else MXQ_TAPS(8);
#undef MXQ_TAPS
}

// ---- convolution over 16 channels, window and pixels resident in LDS ---------------------
// A pixel of 16 channels is one 16-byte piece, and the implicit GEMM brings it into LDS once per tap, with
// an address for each: 140 KB for 128 pixels of a 7 x 7 window and 32 channels out.  Here a work-group
// takes BM consecutive output pixels (in (n, oh, ow) order, regardless of where a row or an image
// ends) and BN output channels, brings the input rows the pixels touch into LDS once, "virtual rows" of
// H + 2 pad an image with pad columns left and right, and all taps of its channels, and forms the
// activation fragments by addresses: two taps of 32 pixels an MFMA, the pixels one behind the other.
// What bounds it is a work-group's one unhidden prologue, 2 to 3 us, and for many columns the weights that
// every work-group brings (25 KB for 7 x 7 and 32 channels), then LDS reads (2 KB an MFMA on 128 pixels, 1.5
// on 256).  Fused, implicit GEMM and this (us): 50176 pixels -> 29, 5 x 5, 9.6 / 6.4, 16928 -> 87, 7 x 7, 11.8 /
// 8.2, 97600 -> 24, 3 x 3, 9.1 / 6.4.  Over more channels, pixels an odd number of pieces apart, it is ahead only
// over 32 into 32 and fewer (200704 -> 32, 3 x 3, 15.0 / 11.7, 83655 -> 17, 5 x 5, 11.2 / 10.8) and level or behind over
// 48 and 64 (11250 -> 11, 5 x 5, 8.4 / 8.4, 200704 -> 64, 3 x 3, 15.1 / 30.9): left at 16.
struct WindowArgs {
  ConvArgs c;
  int pixels_w, rows_h;  // columns of a patch row, virtual rows of an image
  int steps, pitch;      // MFMA steps; 16-byte pieces between the weights of two channels
  int off_patch, off_taps;
};

template <class Cfg>
__global__ __launch_bounds__(256, 2) void conv_window_kernel(WindowArgs t) {
  static_assert(Cfg::WN == 1 && Cfg::kThreads == 256, "four waves below each other");
  constexpr int MI = Cfg::MI, NI = Cfg::NI;
  extern __shared__ __attribute__((aligned(16))) char window_lds[];
  const ConvArgs& p = t.c;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lgrp = lane >> 5;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(window_lds));
  int tm, tn;
  tile_coords(blockIdx.x, (p.M + Cfg::BM - 1) / Cfg::BM, (p.O + Cfg::BN - 1) / Cfg::BN, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN, taps = p.KH * p.KW, plane = p.OH * p.OW;
  // the first virtual row under output pixel m
  auto row_of = [&](int m) {
    const int n = m / plane, oh = (m - n * plane) / p.OW;
    return n * t.rows_h + oh * p.sh;
  };
  const int v0 = row_of(m0);
  {
    const int last = m0 + Cfg::BM < p.M ? m0 + Cfg::BM - 1 : p.M - 1;
    const int pieces = (row_of(last) + (p.KH - 1) * p.dh + 1 - v0) * t.pixels_w;
    const v4i rsrc = make_rsrc(p.data, static_cast<uint32_t>(p.N) * p.H * p.W * 16);
    for (int i = wave * 64; i < pieces; i += 256) {
      const int at = i + lane, row = at / t.pixels_w, v = v0 + row, n = v / t.rows_h;
      const int ih = v - n * t.rows_h - p.ph, iw = at - row * t.pixels_w - p.pw;
      const bool ok = at < pieces && n < p.N &&
                      static_cast<unsigned>(ih) < static_cast<unsigned>(p.H) &&
                      static_cast<unsigned>(iw) < static_cast<unsigned>(p.W);
      dma_buffer(lds0 + t.off_patch + i * 16,
                 ok ? static_cast<uint32_t>(((n * p.H + ih) * p.W + iw) * 16) : kOutOfRange, rsrc);
    }
  }
  {
    const v4i rsrc = make_rsrc(p.weight, static_cast<uint32_t>(p.O) * taps * 16);
    for (int i = wave * 64; i < Cfg::BN * t.pitch; i += 256) {
      const int at = i + lane, o = at / t.pitch, c = at - o * t.pitch;
      const bool ok = o < Cfg::BN && n0 + o < p.O && c < taps;  // zeros meet taps past the last
      dma_buffer(lds0 + i * 16,
                 ok ? static_cast<uint32_t>(((n0 + o) * taps + c) * 16) : kOutOfRange, rsrc);
    }
  }
  int* const tap_at = reinterpret_cast<int*>(window_lds + t.off_taps);
  for (int i = tid; i < 2 * t.steps; i += 256) {
    const int kh = i / p.KW, kw = i - kh * p.KW;
    tap_at[i] = i < taps ? (kh * p.dh * t.pixels_w + kw * p.dw) * 16 : 0;
  }
  const EpiPreOf<kEpiPlain> pre = epi_prefetch<Cfg>(p.epi, n0, p.O);
  const char* pixel[MI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    int m = m0 + wave * Cfg::TM + mi * 32 + lrow;
    m = m < p.M ? m : p.M - 1;  // never stored
    pixel[mi] = window_lds + t.off_patch + ((row_of(m) - v0) * t.pixels_w + m % p.OW * p.sw) * 16;
  }
  const char* const weights = window_lds + (lrow * t.pitch + lgrp) * 16;
  v16i acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll 4
  for (int ks = 0; ks < t.steps; ++ks) {
    const int at = tap_at[2 * ks + lgrp];
    v4i fa[MI], fb[NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) fa[mi] = *reinterpret_cast<const v4i*>(pixel[mi] + at);
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
      fb[ni] = *reinterpret_cast<const v4i*>(weights + (ni * 32 * t.pitch + 2 * ks) * 16);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ni], fa[mi], acc[mi][ni], 0, 0, 0);
  }
  if (blockIdx.x == 0 && tid == 0) epilogue_ranges(p.epi);
  gemm_epilogue_lds<Cfg, EpiScratch<Cfg>::kNeed32>(acc, p.epi, pre, m0, n0, p.M, p.O,
                                                   static_cast<size_t>(p.O),
                                                   reinterpret_cast<v4i*>(window_lds));
}

// The layout of a launch in LDS, and how much of it there is; 0 where the kernel does not take the shape.
template <class Cfg>
size_t window_layout(const ConvArgs& a, WindowArgs& t) {
  const long long data_bytes = static_cast<long long>(a.N) * a.H * a.W * a.C;
  const int taps = a.KH * a.KW;
  if (a.C != 16 || taps < 2 || taps > 64 || a.M <= 0 || data_bytes >= (1LL << 31) ||
      static_cast<long long>(a.O) * taps * 16 >= (1LL << 31) || !aligned16(a.data) ||
      !aligned16(a.weight))
    return 0;
  const long long pixels_w = a.W + 2LL * a.pw, rows_h = a.H + 2LL * a.ph;
  if (a.N * rows_h >= (1LL << 30)) return 0;
  // Most virtual rows under BM consecutive pixels: a step down for every output row they can touch
  // behind the first, a jump for every image.
  const long long down = (Cfg::BM - 2 + a.OW) / a.OW;
  const long long images = (Cfg::BM - 2) / (static_cast<long long>(a.OH) * a.OW) + 1;
  const long long jump = rows_h - static_cast<long long>(a.OH) * a.sh;
  const long long rows = down * a.sh + (a.N > 1 && jump > 0 ? images * jump : 0) +
                         (a.KH - 1LL) * a.dh + 1;
  t.c = a;
  t.steps = (taps + 1) / 2;
  t.pitch = (2 * t.steps) | 1;
  auto up = [](long long pieces) { return (pieces + 63) / 64 * 1024; };  // whole load instructions
  const long long weights = up(static_cast<long long>(Cfg::BN) * t.pitch);
  const long long all = weights + up(rows * pixels_w) + 2 * t.steps * 4;
  if (all > 80 * 1024) return 0;
  t.pixels_w = static_cast<int>(pixels_w);
  t.rows_h = static_cast<int>(rows_h);
  t.off_patch = static_cast<int>(weights);
  t.off_taps = static_cast<int>(all - 2 * t.steps * 4);
  const size_t epilogue = EpiScratch<Cfg>::kNeed32;
  return static_cast<size_t>(all) > epilogue ? static_cast<size_t>(all) : epilogue;
}

typedef GemmCfg<128, 32, 128, 4, 1> CfgWindow;
typedef GemmCfg<256, 32, 128, 4, 1> CfgWindow2;

// Which of the two takes a convolution that the few-tiles kernel does not; 0 for neither.  Up to 32 channels
// out both are ahead of the implicit GEMM, 256 pixels from three tiles of 128 a CU on (us, implicit GEMM, 128,
// 256: 97600 -> 24, 3 x 3, 763 tiles, 9.1 / 6.4 / 6.6, 143748 -> 13, 3 x 3, 1124, 10.4 / 8.3 / 7.7).  More channels
// bring the pixels again for every 32: they pay under windows of 16 taps and more, to two tiles of 128 a CU
// (9604 -> 76, 5 x 5, 225, 7.2 / 5.8, 6075 -> 232, 5 x 5, 384, 7.4 / 6.4), of 256 to six (60984 -> 75, 5 x 5, 1431,
// 12.2 / 12.7 / 11.1, but into int32 20631 -> 393, 7 x 7, 2106, 26.1 / 24.0 / 27.1, 242064 -> 86, 5 x 5, 5676, 35.7 /
// 43.6 / 46.6), and under smaller ones to one (4800 -> 108, 3 x 3, 152, 5.1 / 4.8, but 52983 -> 37, 3 x 3, 828, 7.3 /
// 7.8 / 7.3).  Strided windows read every second piece of LDS and pay from 49 taps on (7605 -> 88, 7 x 7 by 2,
// 9.4 / 7.6, but 25281 -> 37, 5 x 5 by 2 into int32, 7.4 / 8.2).  Where the rows under 256 pixels find no room,
// 128 pixels are not tried, though theirs may (11 images of 40 x 236 -> 20, 7 x 7, 16.6 / 14.4).
int window_cfg(const ConvArgs& a) {
  const int taps = a.KH * a.KW;
  if (a.C != 16 || taps < 9 || (a.sh * a.sw != 1 && taps < 49)) return 0;
  const long cus = num_cus(), t = (a.M + 127L) / 128 * ((a.O + 31) / 32);
  if (a.O <= 32) return t <= 3 * cus ? 66 : 67;
  if (taps < 16) return t <= cus ? 66 : 0;
  return t <= 2 * cus ? 66 : t <= 6 * cus ? 67 : 0;
}

template <class Cfg>
bool launch_window(hipStream_t s, const ConvArgs& a) {
  WindowArgs t;
  const size_t lds = window_layout<Cfg>(a, t);
  if (lds == 0) return false;
  const long tiles =
      static_cast<long>((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.O + Cfg::BN - 1) / Cfg::BN);
  hipLaunchKernelGGL((conv_window_kernel<Cfg>), dim3(static_cast<unsigned>(tiles)), dim3(256), lds,
                     s, t);
  MXQ_LAUNCH_CHECK();
  return true;
}

// ---- 3 x 3 convolution with the input patch resident in LDS -------------------------
// The implicit GEMM above stages every input pixel nine times, once per tap, through the
// CU's 64 bytes per clock from L1 into LDS, which is what bounds every tile below 256 x 256.
// Here a work-group takes 128 consecutive output pixels (in (n, oh, ow) order, regardless
// of where a row or an image ends) and 128 output channels, brings the input rows those
// pixels touch into LDS ONCE -- "virtual rows" n * (H + 2) + ih + 1, so that the zero rows
// above and below an image are rows like any other and a tile that passes from one image
// to the next still reads a contiguous range -- and forms the nine taps' activation
// fragments by address arithmetic: the patch pixel of output pixel (n, oh, ow) under tap
// (kh, kw) is pp0 + kh * (W + 2) + kw.  Only the weights go through the stage ring (128
// rows x 128 bytes per stage: one tap's 128 channels), so a K step moves half the bytes of
// the implicit GEMM's and the ring is half as large: two work-groups of 8 waves share a CU
// and one's loads and epilogue overlap the other's MFMAs.  Stride 1, pad 1, no dilation,
// C a multiple of 128; int8 fused or int32 output through the common epilogue.
constexpr int kPatchBytes = 40 * 1024;   // room for the patch of one tile
#ifdef MXQ_STAMPS
__device__ long long mxq_dbg_stamps[8 * 4096];
#define MXQ_STAMP(k)                                                                  \
  do {                                                                                \
    if (lane == 0 && wave == 0 && blockIdx.x < 4096)                                  \
      mxq_dbg_stamps[blockIdx.x * 8 + (k)] = __builtin_readcyclecounter();            \
  } while (0)
#else
#define MXQ_STAMP(k)
#endif
typedef GemmCfg<128, 128, 128, 4, 2> CfgPatch;  // 8 waves, wave tile 32 pixels x 64 channels

template <int NS>
__global__ __launch_bounds__(512, 2) void conv3x3_patch_kernel(ConvArgs p) {
  typedef CfgPatch Cfg;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, CHW = Cfg::CH;   // CHW: chunks per weight row of a stage
  constexpr int NW = 8, BI = Cfg::B_CHUNKS, KS = Cfg::KS, NI = Cfg::NI;
  constexpr int STAGE_BYTES = BN * BK, RING_BYTES = NS * STAGE_BYTES;
  static_assert(Cfg::MI == 1 && NI == 2 && BI == 2, "wave tile 32 x 64");
  __shared__ __attribute__((aligned(16))) v4i lds[(kPatchBytes + RING_BYTES) / 16];
  char* patch = reinterpret_cast<char*>(lds);
  char* ring = patch + kPatchBytes;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  MXQ_STAMP(4);
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.O + BN - 1) / BN;
  // channel tiles of one pixel tile are neighbours (they share the patch's cache lines)
  const int lid = xcd_remap(blockIdx.x, tiles_m * tiles_n);
  const int tn = lid % tiles_n, tm = lid / tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  const int PW = p.W + 2, CH = p.C >> 4;   // patch pixels per row, 16-byte chunks per pixel
  const int ohow = p.OH * p.OW;

  // the range of virtual rows this tile touches
  const int ma = m0, mb = (m0 + BM - 1 < p.M) ? m0 + BM - 1 : p.M - 1;
  const int na = ma / ohow, oha = (ma - na * ohow) / p.OW;
  const int nb = mb / ohow, ohb = (mb - nb * ohow) / p.OW;
  const int vr0 = na * (p.H + 2) + oha;
  const int rows = nb * (p.H + 2) + ohb + 2 - vr0 + 1;

  // The patch: a row of it is RP pixels (the W + 2 real ones padded so that a row is whole
  // load instructions of 64 slots: the row of an instruction is then wave-uniform and no lane
  // divides anything), chunk j of patch pixel pp at slot pp * CH + (j ^ patch_swz(pp)).  A
  // fragment read is 16 consecutive pixels per LDS pass; with 128-byte pixels two of them
  // fill the banks once, so the XOR advances every second pixel, with wider pixels every one.
  const int ch_shift = __builtin_ctz(CH);
  const int per_row = (PW * CH + 63) >> 6;        // load instructions per patch row
  const int RP = (per_row << 6) >> ch_shift;      // pixels per patch row
  const int swz_shift = CH == 8 ? 1 : 0;
  auto patch_swz = [&](int pixel) { return (pixel >> swz_shift) & (CH - 1); };
  {
    const v4i rsrc = make_rsrc(p.data, static_cast<uint32_t>(p.N) * p.H * p.W * p.C);
    const uint32_t patch_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(patch));
    const int instrs = rows * per_row;
    for (int it = wave; it < instrs; it += NW) {
      const int r = it / per_row, part = it - r * per_row;    // wave-uniform
      const int vabs = vr0 + r;
      const int n = vabs / (p.H + 2), ih = vabs - n * (p.H + 2) - 1;
      const bool row_ok = n < p.N && static_cast<unsigned>(ih) < static_cast<unsigned>(p.H);
      const int q = part * 64 + lane;                          // slot inside the row
      const int px = q >> ch_shift, pp = r * RP + px;
      const int j = (q & (CH - 1)) ^ patch_swz(pp);
      const int iw = px - 1;
      const bool ok = row_ok && static_cast<unsigned>(iw) < static_cast<unsigned>(p.W);
      const uint32_t off =
          ok ? static_cast<uint32_t>(((n * p.H + ih) * p.W + iw) * p.C + 16 * j) : kOutOfRange;
      dma_buffer(patch_addr + it * 1024, off, rsrc);
    }
  }
  // the weights: stage s = tap s / (C / BK), channel block s % (C / BK); OHWI rows are K-contiguous
  RowIssuerBuffer<Cfg, BI> bi;
  bi.init(p.weight, n0, p.O, p.K, wave, lane, 0);
  const uint32_t ring_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));
  const int KT = p.K / BK;
  auto issue = [&](int stage) {
    if (stage >= KT) return;
    const uint32_t sb = ring_addr + static_cast<uint32_t>(stage % NS) * STAGE_BYTES;
#pragma unroll
    for (int j = 0; j < BI; ++j) bi.issue(j, stage, sb + (j * NW + wave) * 1024);
  };
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) issue(st);
  MXQ_STAMP(5);
  EpiPreOf<kEpiPlain> pre = epi_prefetch<Cfg>(p.epi, n0, p.O);
  MXQ_STAMP(6);

  // this lane's output pixel and its patch pixel under tap (0, 0)
  const int frow = lane & 31, fgrp = lane >> 5;
  int m = m0 + wm * Cfg::TM + frow;
  m = m < p.M ? m : p.M - 1;   // rows past the end repeat the last pixel; never stored
  const int n = m / ohow, rem = m - n * ohow;
  const int oh = rem / p.OW, ow = rem - oh * p.OW;
  const int pp0 = (n * (p.H + 2) + oh - vr0) * RP + ow;
  const int rb = wn * Cfg::TN + frow;
  int fb0[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) fb0[ks] = rb * CHW + ((ks * 2 + fgrp) ^ swz<CHW>(rb));

  v16i acc[1][NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[0][ni][v] = 0;

  const int blocks = p.C / BK;   // stages per tap
  int tap = 0, cblk = 0, pp = pp0;   // of the stage computed next
  MXQ_STAMP(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the patch and the first stages
  MXQ_STAMP(1);
  for (int kt = 0; kt < KT; ++kt) {
    if (kt > 0) {
      const int newest = (kt + NS - 2) < (KT - 1) ? (kt + NS - 2) : (KT - 1);
      wait_ahead<BI, NS - 2>(newest - kt);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // ... and what it read of stage kt - 1
    __builtin_amdgcn_s_barrier();
    issue(kt + NS - 1);
    const v4i* sbw = reinterpret_cast<const v4i*>(ring + (kt % NS) * STAGE_BYTES);
    const v4i* pix = reinterpret_cast<const v4i*>(patch) + pp * CH;
    const int sw_ = patch_swz(pp);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const v4i fa = pix[(cblk * (BK / 16) + ks * 2 + fgrp) ^ sw_];
      v4i fb[NI];
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) fb[ni] = sbw[fb0[ks] + ni * 32 * CHW];
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[0][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ni], fa, acc[0][ni], 0, 0, 0);
    }
    if (++cblk == blocks) {
      cblk = 0;
      ++tap;
      const int kh = tap / 3, kw = tap - 3 * kh;
      pp = pp0 + kh * RP + kw;
    }
  }
  MXQ_STAMP(2);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (blockIdx.x == 0 && tid == 0) epilogue_ranges(p.epi);
  gemm_epilogue_lds<Cfg, kPatchBytes + RING_BYTES>(acc, p.epi, pre, m0, n0, p.M, p.O,
                                                   static_cast<size_t>(p.O), lds);
  MXQ_STAMP(3);
}

#ifdef MXQ_STAMPS
extern "C" int mxq_dbg_read_stamps(long long* host, int count) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(mxq_dbg_stamps), sizeof(long long) * count) ==
                 hipSuccess
             ? 0
             : -1;
}
#endif

// Virtual rows the patch of a 128-pixel tile can span: the rows its pixels lie in, one
// above, one below, and two halo rows for every image boundary inside the tile.
inline int conv3x3_patch_rows(int OH, int OW) {
  const int out_rows = (128 + OW - 2) / OW + 1;
  const int crossings = (128 + OH * OW - 2) / (OH * OW);
  return out_rows + 2 + 2 * crossings;
}

bool conv3x3_patch_ok(const ConvArgs& a) {
  const long long data_bytes = static_cast<long long>(a.N) * a.H * a.W * a.C;
  const int ch = a.C / 16;
  return a.KH == 3 && a.KW == 3 && a.sh == 1 && a.sw == 1 && a.ph == 1 && a.pw == 1 &&
         a.dh == 1 && a.dw == 1 && a.C % 128 == 0 && (ch & (ch - 1)) == 0 && a.O % 16 == 0 &&
         aligned16(a.data) && aligned16(a.weight) && data_bytes < (1LL << 31) &&
         static_cast<long long>(a.O) * a.K < (1LL << 31) &&
         // (a patch row is whole load instructions of 1 KiB)
         static_cast<long long>(conv3x3_patch_rows(a.OH, a.OW)) *
                 (((a.W + 2) * ch + 63) / 64 * 1024) <=
             kPatchBytes;
}

void launch_conv3x3_patch(hipStream_t s, const ConvArgs& a) {
  const long tiles = static_cast<long>((a.M + 127) / 128) * ((a.O + 127) / 128);
  hipLaunchKernelGGL(conv3x3_patch_kernel<2>, dim3(static_cast<unsigned>(tiles)), dim3(512), 0, s,
                     a);
  MXQ_LAUNCH_CHECK();
}

typedef GemmCfg<256, 256, 64, 2, 4> CfgL8;   // 8 waves, wave tile 128 x 64
typedef GemmCfg<256, 128, 64, 4, 2> CfgW128; // 8 waves, wave tile 64 x 64
typedef GemmCfg<256, 64, 64, 4, 1> CfgW64;   // 4 waves, wave tile 64 x 64
typedef GemmCfg<128, 128, 64, 2, 2> CfgM;    // 4 waves, wave tile 64 x 64
typedef GemmCfg<64, 64, 64, 2, 2> CfgS;      // 4 waves, wave tile 32 x 32
typedef GemmCfg<256, 256, 64, 2, 2> CfgL4;   // 4 waves, wave tile 128 x 128
// 128-byte stages: half as many K steps
typedef GemmCfg<256, 256, 128, 2, 4> CfgL8K;
typedef GemmCfg<256, 128, 128, 4, 2> CfgW128K;
typedef GemmCfg<128, 128, 128, 2, 2> CfgMK;
typedef GemmCfg<64, 64, 128, 2, 2> CfgSK;
typedef GemmCfg<128, 64, 128, 2, 2> CfgRK;
typedef GemmCfg<64, 128, 128, 2, 2> CfgQK;
typedef GemmCfg<64, 64, 256, 2, 2> CfgSK2;
typedef GemmCfg<128, 32, 128, 4, 1> CfgNK;

template <class Cfg, int NS, int PIPE>
void launch_dma(hipStream_t s, ConvArgs a, int splits, const Workspace& ws) {
  const long tiles =
      static_cast<long>((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.O + Cfg::BN - 1) / Cfg::BN);
  splitk_setup<Cfg>(s, a.sk, tiles, a.K, splits, ws.ptr, ws.bytes);
  hipLaunchKernelGGL((conv_dma_kernel<Cfg, NS, PIPE>),
                     dim3(static_cast<unsigned>(tiles * a.sk.splits)), dim3(Cfg::kThreads), 0, s,
                     a);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg, int NS>
void launch_sliced(hipStream_t s, ConvArgs a, int splits, const Workspace& ws) {
  const long tiles =
      static_cast<long>((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.O + Cfg::BN - 1) / Cfg::BN);
  splitk_setup<typename Cfg::Tile>(s, a.sk, tiles, a.K, splits, ws.ptr, ws.bytes);
  hipLaunchKernelGGL((conv_sliced_kernel<Cfg, NS>),
                     dim3(static_cast<unsigned>(tiles * a.sk.splits)), dim3(Cfg::kThreads), 0, s,
                     a);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg>
void launch_pair(hipStream_t s, const ConvArgs& a, const ConvArgs& b) {
  auto tiles = [](const ConvArgs& x) {
    return static_cast<long>((x.M + Cfg::BM - 1) / Cfg::BM) * ((x.O + Cfg::BN - 1) / Cfg::BN);
  };
  const ConvPair p = {a, b, static_cast<int>(tiles(a))};
  hipLaunchKernelGGL((conv_pair_kernel<Cfg, 2>), dim3(static_cast<unsigned>(tiles(a) + tiles(b))),
                     dim3(Cfg::kThreads), 0, s, p);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg>
void launch_cfg(hipStream_t s, const ConvArgs& a, bool aligned) {
  const int tiles = ((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.O + Cfg::BN - 1) / Cfg::BN);
  if (aligned)
    hipLaunchKernelGGL((conv_kernel<Cfg, true>), dim3(tiles), dim3(Cfg::kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((conv_kernel<Cfg, false>), dim3(tiles), dim3(Cfg::kThreads), 0, s, a);
  MXQ_LAUNCH_CHECK();
}

// ---- layout adapters ------------------------------------------------------------
// A transpose [B][R][S] -> [B][S][RP] of bytes, 16 | RP, zeros in positions R ... RP - 1, that asks
// nothing of R, S or the input's address: a lane gathers 16 bytes S apart and stores them as one
// piece.  The lanes run along S, so that a load instruction of a wave reads whole lines, whatever S is
// (along the pieces of a row, as it was, it read 64 lines for 64 bytes: the weights of 7 x 7 x 512
// -> 512, 3 x 3).  Where a row has four pieces and more, the four waves of a work-group take four of
// them, 64 bytes that leave through one L2.
// Two of them fit a launch, or one rides along in another's: the weights of a convolution
// ([O][C][taps] -> [O][taps][C]) next to its data.  A launch of its own costs 4.6-5.9 us inside a
// network however little it moves (launch, then a cold round trip to memory).
struct GatherJob {
  const uint8_t* in;
  uint8_t* out;
  int R, S, RP;
  unsigned tiles_s, tiles_k;  // of 64 columns and 4 pieces; 0: pieces one behind the other
  unsigned pieces;            // B * S * RP / 16, or what covers it in tiles
  unsigned blocks;            // work-groups' worth of pieces; 0: no job
  // of the two extents that a place is divided by: tiles_s and tiles_k, or S and the pieces of a row
  unsigned magic_s, magic_k;
};

// work-groups a riding job gets: enough to be done when the carrier is
__host__ __device__ inline unsigned job_blocks(const GatherJob& job) {
  return job.blocks < 1024u ? job.blocks : 1024u;
}

GatherJob no_job() { return GatherJob{nullptr, nullptr, 0, 1, 16, 0, 0, 0, 0, 0, 0}; }

// floor(n / d) for n < 2^31, magic = 2^31 / d + 1: the product is at most one too large.  (A division
// by a value that the compiler does not know is a dozen instructions.  A launch of a few work-groups
// waits for its rider, 37 x 32 x 9 weights beside 5 images of 12 x 12: 3.12 us with the divisions and
// all pieces clamped, 2.96 without the clamping, 2.80 without both.)
unsigned gather_magic(unsigned d) { return static_cast<unsigned>((1ull << 31) / d + 1); }
__device__ __forceinline__ unsigned gather_quotient(unsigned n, unsigned d, unsigned magic) {
  const unsigned q = __umulhi(2u * n + 1u, magic);
  return q - (q * d > n);
}

bool gather_job_ok(const void* out, long long B, long long S, long long RP) {
  return RP % 16 == 0 && aligned16(out) && B * S * RP > 0 &&
         B * (S + 64) * (RP / 16 + 4) < (1LL << 31);
}
GatherJob gather_job(const void* in, void* out, int B, int R, int S, int RP) {
  GatherJob j = {static_cast<const uint8_t*>(in), static_cast<uint8_t*>(out), R, S, RP, 0, 0, 0, 0, 0, 0};
  const unsigned per_row = static_cast<unsigned>(RP) >> 4;
  if (S >= 64 && per_row >= 4) {
    j.tiles_s = (static_cast<unsigned>(S) + 63u) / 64u;
    j.tiles_k = (per_row + 3u) / 4u;
    j.blocks = static_cast<unsigned>(B) * j.tiles_s * j.tiles_k;
    j.pieces = j.blocks * 256u;
    j.magic_s = gather_magic(j.tiles_s);
    j.magic_k = gather_magic(j.tiles_k);
  } else {
    j.pieces = static_cast<unsigned>(B) * static_cast<unsigned>(S) * per_row;
    j.blocks = (j.pieces + 255u) / 256u;
    j.magic_s = gather_magic(static_cast<unsigned>(S));
    j.magic_k = gather_magic(per_row);
  }
  return j;
}

__device__ __forceinline__ void gather_job_run(const GatherJob& j, unsigned block,
                                               unsigned nblocks) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const unsigned per_row = static_cast<unsigned>(j.RP) >> 4, S = static_cast<unsigned>(j.S);
  for (unsigned item = block; item < j.blocks; item += nblocks) {
    unsigned b, k, s;
    if (j.tiles_s != 0) {
      const unsigned rest = gather_quotient(item, j.tiles_s, j.magic_s);
      b = gather_quotient(rest, j.tiles_k, j.magic_k);
      s = (item - rest * j.tiles_s) * 64u + (threadIdx.x & 63u);
      k = (rest - b * j.tiles_k) * 4u + (threadIdx.x >> 6);
      if (s >= S || k >= per_row) continue;
    } else {
      const unsigned t = item * 256u + threadIdx.x;
      if (t >= j.pieces) continue;
      const unsigned rest = gather_quotient(t, S, j.magic_s);
      s = t - rest * S;
      b = gather_quotient(rest, per_row, j.magic_k);
      k = rest - b * per_row;
    }
    const int rows = j.R - static_cast<int>(16 * k);  // of the input under this piece
    const uint8_t* src = j.in + (static_cast<size_t>(b) * j.R + (rows > 0 ? 16 * k : 0)) * S + s;
    uint32_t w[4] = {0, 0, 0, 0};
    // whole pieces without the clamping (64 x 16 x 113 x 113 9.6 -> 7.2 us), where all lanes have them
    if (__all(rows >= 16)) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        w[i >> 2] |= static_cast<uint32_t>(src[static_cast<size_t>(i) * S]) << (8 * (i & 3));
    } else {
      const int last = rows > 0 ? rows - 1 : 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t x = src[static_cast<size_t>(i < last ? i : last) * S];
        w[i >> 2] |= (i < rows ? x : 0u) << (8 * (i & 3));
      }
    }
    *reinterpret_cast<u4*>(j.out + (static_cast<size_t>(b) * S + s) * j.RP + 16 * k) =
        u4{w[0], w[1], w[2], w[3]};
  }
}

// Batched transpose [B][R][S] -> [B][S][RP] through a padded LDS tile; reads are
// contiguous along S, writes contiguous along R.  RP >= R: positions R..RP-1 of every
// output row are written as zeros (channel padding).
template <typename T>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ in,
                                                        T* __restrict__ out, int R, int S,
                                                        int RP) {
  __shared__ T tile[64][65];
  const size_t b = blockIdx.z;
  const int r0 = blockIdx.y * 64, s0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const T* src = in + b * static_cast<size_t>(R) * S;
  T* dst = out + b * static_cast<size_t>(RP) * S;
  for (int i = ty; i < 64; i += 4) {
    const int r = r0 + i, s = s0 + tx;
    tile[i][tx] = (r < R && s < S) ? src[static_cast<size_t>(r) * S + s] : T(0);
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int s = s0 + i, r = r0 + tx;
    if (r < RP && s < S) dst[static_cast<size_t>(s) * RP + r] = tile[tx][i];
  }
}

// The byte form of the same transpose for friendly shapes (S % 4 == 0, RP % 16 == 0,
// aligned pointers): a work-group takes 64 rows x 128 columns, every thread loads dwords
// along S (a wave reads whole 128-byte runs), transposes 4 x 4 bytes in registers with
// v_perm and parks the result in LDS, from where 16-byte pieces of the output rows leave
// (a wave writes 1 KiB contiguous when the group covers all RP positions of its rows).
__global__ __launch_bounds__(256) void transpose_i8_kernel(const uint8_t* __restrict__ in,
                                                           uint8_t* __restrict__ out, int R,
                                                           int S, int RP, int B, GatherJob job,
                                                           unsigned riders) {
  constexpr int kPitch = 17;  // dwords per transposed row: 64 bytes + 4 of padding
  __shared__ uint32_t tile[128 * kPitch];
  if (static_cast<int>(blockIdx.z) >= B) {   // the extra z slices carry the riding job
    const unsigned wide = (S + 127) >> 7, high = (RP + 63) >> 6;
    gather_job_run(job, ((blockIdx.z - B) * high + blockIdx.y) * wide + blockIdx.x, riders);
    return;
  }
  const size_t b = blockIdx.z;
  const int r0 = blockIdx.y * 64, s0 = blockIdx.x * 128;
  const int t = threadIdx.x;
  const uint8_t* src = in + b * static_cast<size_t>(R) * S;
  uint8_t* dst = out + b * static_cast<size_t>(RP) * S;
  const int sq = t & 31;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int rq = (t >> 5) + 8 * pass;
    const int s = s0 + 4 * sq;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = r0 + 4 * rq + j;
      w[j] = (r < R && s < S)
                 ? *reinterpret_cast<const uint32_t*>(src + static_cast<size_t>(r) * S + s)
                 : 0u;
    }
    // x[i] = byte i of w[0..3]
    const uint32_t t0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    tile[(4 * sq + 0) * kPitch + rq] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    tile[(4 * sq + 1) * kPitch + rq] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    tile[(4 * sq + 2) * kPitch + rq] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    tile[(4 * sq + 3) * kPitch + rq] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
  }
  __syncthreads();
  const int nb = min(64, RP - r0);  // bytes of every output row this group owns (16 | nb)
  const int per_row = nb >> 4;      // 16-byte pieces per row: 1..4
  const int pieces = 128 * per_row;
  for (int c = t; c < pieces; c += 256) {
    const int sl = per_row == 4 ? (c >> 2) : (per_row == 2 ? (c >> 1) : (per_row == 1 ? c : c / 3));
    const int k = c - sl * per_row;
    if (s0 + sl >= S) continue;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    u4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = tile[sl * kPitch + 4 * k + i];
    *reinterpret_cast<u4*>(dst + static_cast<size_t>(s0 + sl) * RP + r0 + 16 * k) = v;
  }
}

// The same on 128 rows x 128 columns with 16-byte loads (S % 16 == 0, S and RP >= 128,
// 16-byte aligned input as well): a thread takes 16 bytes along S of four consecutive rows, four load
// instructions instead of sixteen, and the output runs are whole 128-byte lines.
struct WideOrder {
  unsigned tiles_s, tiles_r, total, per_xcd;
  unsigned grid;   // work-groups of the tile grid
};

template <int PIECE>
__global__ __launch_bounds__(256) void transpose_i8_wide_kernel(const uint8_t* __restrict__ in,
                                                                uint8_t* __restrict__ out,
                                                                int R, int S, int RP,
                                                                WideOrder o, GatherJob job) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  constexpr int kPitch = 33;  // dwords per transposed row: 128 bytes + 4 of padding
  __shared__ uint32_t tile[128 * kPitch];
  if (blockIdx.x >= o.grid) {   // blocks past the tile grid carry the riding job
    gather_job_run(job, blockIdx.x - o.grid, job_blocks(job));
    return;
  }
  // the tile sequence runs along S first, then R, then the batch; with o.per_xcd != 0 the
  // round-robin of work-group ids over the 8 XCDs is undone, so that every XCD owns a
  // contiguous range of it and tiles that share input cache lines meet in one L2
  unsigned item = blockIdx.x;
  if (o.per_xcd != 0) {
    item = (blockIdx.x & 7u) * o.per_xcd + (blockIdx.x >> 3);
    if (item >= o.total) return;
  }
  const unsigned rest = item / o.tiles_s, ts = item - rest * o.tiles_s;
  const unsigned bq = rest / o.tiles_r, tr = rest - bq * o.tiles_r;
  const size_t b = bq;
  const int r0 = tr * 128, s0 = ts * 128;
  const int t = threadIdx.x;
  const uint8_t* src = in + b * static_cast<size_t>(R) * S;
  uint8_t* dst = out + b * static_cast<size_t>(RP) * S;
  const int sq = t & 7, rq = t >> 3;
  const int s = s0 + 16 * sq;
  u4 w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = r0 + 4 * rq + j;
    w[j] = (r < R && s < S) ? __builtin_nontemporal_load(reinterpret_cast<const u4*>(
                                  src + static_cast<size_t>(r) * S + s))
                            : u4{0, 0, 0, 0};
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    // x[i] = byte i of w[0..3][d]
    const uint32_t t0 = __builtin_amdgcn_perm(w[1][d], w[0][d], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(w[1][d], w[0][d], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(w[3][d], w[2][d], 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(w[3][d], w[2][d], 0x07030602u);
    const int row = 16 * sq + 4 * d;
    tile[(row + 0) * kPitch + rq] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    tile[(row + 1) * kPitch + rq] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    tile[(row + 2) * kPitch + rq] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    tile[(row + 3) * kPitch + rq] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
  }
  __syncthreads();
  const int nb = min(128, RP - r0);  // bytes of every output row this group owns (PIECE | nb)
  const int per_row = nb / PIECE;
  const int pieces = 128 * per_row;
  for (int c = t; c < pieces; c += 256) {
    const int sl = per_row == 128 / PIECE ? c / (128 / PIECE) : c / per_row;
    const int k = c - sl * per_row;
    if (s0 + sl < S) {
      uint8_t* to = dst + static_cast<size_t>(s0 + sl) * RP + r0 + PIECE * k;
      if (PIECE == 16) {
        u4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = tile[sl * kPitch + 4 * k + i];
        __builtin_nontemporal_store(v, reinterpret_cast<u4*>(to));
      } else {
        // rows of 4 | RP bytes (14 x 14 planes): dword pieces, a wave still writes whole runs
        __builtin_nontemporal_store(tile[sl * kPitch + k], reinterpret_cast<uint32_t*>(to));
      }
    }
  }
}

__global__ __launch_bounds__(256) void copy16_kernel(const uint8_t* __restrict__ in,
                                                     uint8_t* __restrict__ out, size_t pieces) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const size_t stride = static_cast<size_t>(gridDim.x) * 256;
  for (size_t q = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; q < pieces; q += stride)
    reinterpret_cast<u4*>(out)[q] = reinterpret_cast<const u4*>(in)[q];
}

// Whatever the kernels above do not take, up to two jobs per launch.
__global__ __launch_bounds__(256) void gather_transpose_kernel(GatherJob first, GatherJob second) {
  if (blockIdx.x < first.blocks)
    gather_job_run(first, blockIdx.x, first.blocks);
  else
    gather_job_run(second, blockIdx.x - first.blocks, job_blocks(second));
}

// A thin extent (at most 64 bytes, e.g. 7 x 7 planes) beside a long one that is a multiple of
// 128: see thin_transpose_tile.  One matrix per blockIdx.y.
template <bool THIN_IN>
__global__ __launch_bounds__(256) void transpose_i8_thin_kernel(const uint8_t* __restrict__ in,
                                                                uint8_t* __restrict__ out,
                                                                int L, int T) {
  __shared__ __attribute__((aligned(16))) uint8_t flat[128 * 64];
  const size_t plane = static_cast<size_t>(L) * T;
  thin_transpose_tile<THIN_IN>(in + blockIdx.y * plane, out + blockIdx.y * plane, L, T,
                               blockIdx.x * 128, flat);
}

// Space-to-depth by 2 while going from planes to pixels: out[b][h2][w2][(dh*2+dw)*C + c] =
// in[b][c][2*h2 - off_h + dh][2*w2 - off_w + dw] (zero outside the plane), the channel run
// of every output pixel zero-padded to CP bytes.  A stride-2 convolution over few channels
// becomes a unit-stride one over 4*C channels and half the window, which suits the
// direct-to-LDS kernels (16-byte channel runs) far better than 3 or 4 channels do.
__global__ __launch_bounds__(256) void s2d_nhwc_kernel(const int8_t* __restrict__ in,
                                                       int8_t* __restrict__ out, int C, int H,
                                                       int W, int H2, int W2, int off_h,
                                                       int off_w, int CP, size_t pixels) {
  for (size_t p = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; p < pixels;
       p += static_cast<size_t>(gridDim.x) * 256) {
    const int w2 = static_cast<int>(p % W2);
    const size_t t = p / W2;
    const int h2 = static_cast<int>(t % H2);
    const size_t b = t / H2;
    const int8_t* img = in + b * static_cast<size_t>(C) * H * W;
    int8_t* dst = out + p * CP;
    for (int d = 0; d < 4; ++d) {
      const int h = 2 * h2 - off_h + (d >> 1), w = 2 * w2 - off_w + (d & 1);
      const bool inside = static_cast<unsigned>(h) < static_cast<unsigned>(H) &&
                          static_cast<unsigned>(w) < static_cast<unsigned>(W);
      for (int c = 0; c < C; ++c)
        dst[d * C + c] = inside ? img[(static_cast<size_t>(c) * H + h) * W + w] : int8_t(0);
    }
    for (int c = 4 * C; c < CP; ++c) dst[c] = 0;
  }
}

// Input rows that do not start on 128-byte marks (56 x 56 and 28 x 28 planes on the way to
// pixels) share cache lines between neighbouring tiles along S: there the round-robin of
// work-group ids over the XCDs is undone (64 x 256 x 56 x 56: 22.6 -> 21.1 us, 64 x 512 x 28 x 28:
// 14.3 -> 12.1 us).  Rows on the marks lose 10 % that way (64 x 64 planes: 25.6 -> 28.9 us) and
// the way back to planes gains nothing reliably, so those keep the plain order.

template <int PIECE>
void launch_wide(hipStream_t s, const void* in, void* out, int B, int R, int S, int RP,
                 const GatherJob& job) {
  WideOrder o;
  o.tiles_s = static_cast<unsigned>((S + 127) / 128);
  o.tiles_r = static_cast<unsigned>((RP + 127) / 128);
  const unsigned long long total = 1ull * o.tiles_s * o.tiles_r * static_cast<unsigned>(B);
  MXQ_CHECK(total < (1ull << 31) - 256, "transpose grid too large");
  o.total = static_cast<unsigned>(total);
  o.per_xcd = (S % 128 != 0) ? (o.total + 7u) / 8u : 0u;
  o.grid = o.per_xcd != 0 ? o.per_xcd * 8u : o.total;
  hipLaunchKernelGGL(transpose_i8_wide_kernel<PIECE>, dim3(o.grid + job_blocks(job)), dim3(256), 0,
                     s, static_cast<const uint8_t*>(in), static_cast<uint8_t*>(out), R, S, RP, o,
                     job);
  MXQ_LAUNCH_CHECK();
}

// [B][R][S] -> [B][S][RP].  `rider`, when given, is a job the launch carries along if
// its kernel can (then rider->blocks is cleared); the caller launches what is left.
template <typename T>
void launch_transpose(hipStream_t s, const void* in, void* out, int B, int R, int S, int RP,
                      GatherJob* rider = nullptr) {
  if (B == 0 || RP == 0 || S == 0) return;
  MXQ_CHECK(RP >= R, "padded extent below the extent");
  const GatherJob job = rider != nullptr ? *rider : no_job();
  auto carried = [&]() {
    if (rider != nullptr) rider->blocks = 0;
  };
  auto gather = [&]() {
    const GatherJob me = gather_job(in, out, B, R, S, RP);
    hipLaunchKernelGGL(gather_transpose_kernel, dim3(me.blocks + job_blocks(job)), dim3(256), 0, s,
                       me, job);
    MXQ_LAUNCH_CHECK();
    carried();
  };
  const bool gathers = sizeof(T) == 1 && R > 0 && gather_job_ok(out, B, S, RP);
  // only the kernels that put batches and row tiles on grid.y / grid.z have their limit
  auto check_yz = [&]() {
    MXQ_CHECK(B < 65535 && (RP + 63) / 64 <= 65535, "transpose grid too large");
  };
  if (sizeof(T) == 1 && S % 16 == 0 && S >= 128 && RP >= 128 && RP % 4 == 0 && RP % 16 != 0 &&
      aligned16(in) && (reinterpret_cast<uintptr_t>(out) & 3u) == 0) {
    launch_wide<4>(s, in, out, B, R, S, RP, job);
    carried();
    return;
  }
  if (sizeof(T) == 1 && S % 4 == 0 && RP % 16 == 0 &&
      (reinterpret_cast<uintptr_t>(in) & 3u) == 0 && aligned16(out)) {
    // (with fewer than 128 columns half of the wide tile's lanes would idle: 64 x 56 x 56 x 64
    // back to planes takes 7.8 us that way against 6.0 us)
    if (S % 16 == 0 && S >= 128 && RP >= 128 && aligned16(in)) {
      launch_wide<16>(s, in, out, B, R, S, RP, job);
      carried();
      return;
    }
    check_yz();
    const unsigned per_z = static_cast<unsigned>((S + 127) / 128) * ((RP + 63) / 64);
    const unsigned extra_z = (job_blocks(job) + per_z - 1) / per_z;
    const bool fits = B + extra_z <= 65535u;  // the rider, else a launch of its own
    dim3 grid128((S + 127) / 128, (RP + 63) / 64, fits ? B + extra_z : B);
    hipLaunchKernelGGL(transpose_i8_kernel, grid128, dim3(256), 0, s,
                       static_cast<const uint8_t*>(in), static_cast<uint8_t*>(out), R, S, RP, B,
                       job, fits ? extra_z * per_z : 0u);
    MXQ_LAUNCH_CHECK();
    if (fits) carried();
    return;
  }
  if (gathers && S > 1 && S <= 64 && static_cast<long long>(B) * RP * S <= (4LL << 20)) {
    // a small tensor with a thin inner extent (3 x 3 weights, 7 x 7 planes)
    gather();
    return;
  }
  if (sizeof(T) == 1 && RP == R && aligned16(in) && aligned16(out)) {
    // a thin extent (<= 64) beside a long one that is a multiple of 128
    const bool thin_in = S <= 64 && R % 128 == 0;
    const bool thin_out = R <= 64 && S % 128 == 0;
    if ((thin_in && S == 1) || (thin_out && R == 1)) {
      // a thin extent of 1 (the weights of a 1 x 1 convolution): the transpose is a copy
      const size_t pieces = static_cast<size_t>(B) * R * S / 16;  // 128 | R * S
      const size_t want = (pieces + 255) / 256;
      const size_t cap = static_cast<size_t>(num_cus()) * 8;
      hipLaunchKernelGGL(copy16_kernel, dim3(static_cast<unsigned>(want < cap ? want : cap)),
                         dim3(256), 0, s, static_cast<const uint8_t*>(in),
                         static_cast<uint8_t*>(out), pieces);
      MXQ_LAUNCH_CHECK();
      return;
    }
    if (thin_in || thin_out) {
      const int L = thin_in ? R : S, thin = thin_in ? S : R;
      MXQ_CHECK(B <= 65535, "transpose grid too large");
      dim3 grid(L / 128, B);
      if (thin_in)
        hipLaunchKernelGGL(transpose_i8_thin_kernel<true>, grid, dim3(256), 0, s,
                           static_cast<const uint8_t*>(in), static_cast<uint8_t*>(out), L, thin);
      else
        hipLaunchKernelGGL(transpose_i8_thin_kernel<false>, grid, dim3(256), 0, s,
                           static_cast<const uint8_t*>(in), static_cast<uint8_t*>(out), L, thin);
      MXQ_LAUNCH_CHECK();
      return;
    }
  }
  if (gathers) {
    gather();
    return;
  }
  check_yz();
  dim3 grid((S + 63) / 64, (RP + 63) / 64, B);
  hipLaunchKernelGGL((transpose_kernel<T>), grid, dim3(256), 0, s, static_cast<const T*>(in),
                     static_cast<T*>(out), R, S, RP);
  MXQ_LAUNCH_CHECK();
}

// Output tile of a direct-to-LDS configuration of this file (what a split-K work-group
// leaves in the workspace); false for the register-staged ones.
bool conv_cfg_tile(int cfg, int& bm, int& bn) {
  switch (cfg) {
    case 11: case 16: case 35: bm = 256; bn = 256; return true;
    case 12: case 22: case 36: bm = 256; bn = 128; return true;
    case 13: case 23: bm = 256; bn = 64; return true;
    case 14: case 24: case 33: case 34: bm = 128; bn = 128; return true;
    case 15: case 25: case 31: case 32: case 39: bm = 64; bn = 64; return true;
    case 37: bm = 128; bn = 64; return true;
    case 38: bm = 64; bn = 128; return true;
    case 40: bm = 64; bn = 64; return true;
    case 41: case 42: bm = 128; bn = 32; return true;
    case 43: bm = 128; bn = 128; return true;
    default: return false;
  }
}

struct ConvGeometry {
  int N, H, W, C, O, KH, KW, sh, sw, ph, pw, dh, dw;
  int OH, OW;
  long long M, K;
  bool is_fc;  // 1x1, unit stride, no padding: the FC of the flattened pixels
};

ConvGeometry conv_geometry(int N, int H, int W, int C, int O, int KH, int KW, int stride_h,
                           int stride_w, int pad_h, int pad_w, int dilate_h, int dilate_w) {
  MXQ_CHECK(N >= 0 && H > 0 && W > 0 && C > 0 && O > 0 && KH > 0 && KW > 0, "bad shape");
  MXQ_CHECK(stride_h > 0 && stride_w > 0 && dilate_h > 0 && dilate_w > 0 && pad_h >= 0 &&
                pad_w >= 0,
            "bad stride/dilate/pad");
  const int eh = dilate_h * (KH - 1) + 1, ew = dilate_w * (KW - 1) + 1;
  MXQ_CHECK(H + 2 * pad_h >= eh && W + 2 * pad_w >= ew, "kernel larger than padded input");
  ConvGeometry g = {N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w, dilate_h, dilate_w,
                    0, 0, 0, 0, false};
  g.OH = (H + 2 * pad_h - eh) / stride_h + 1;
  g.OW = (W + 2 * pad_w - ew) / stride_w + 1;
  g.M = static_cast<long long>(N) * g.OH * g.OW;
  g.K = static_cast<long long>(KH) * KW * C;
  MXQ_CHECK(g.M < (1LL << 31) && g.K < (1LL << 31), "problem too large for 32-bit tile indices");
  g.is_fc = KH == 1 && KW == 1 && stride_h == 1 && stride_w == 1 && pad_h == 0 && pad_w == 0;
  return g;
}

struct ConvPlan {
  int cfg;
  int splits;
};

// What conv_nhwc would launch for a convolution that does not reduce to the FC.  `aligned`:
// C % 16 == 0 and 16-byte aligned operands.
ConvPlan plan_conv(const ConvGeometry& g, bool aligned, const GemmForce& force) {
  ConvPlan plan = {force.cfg, force.splits};
  const int M = static_cast<int>(g.M), K = static_cast<int>(g.K), O = g.O;
  const long long data_bytes = static_cast<long long>(g.N) * g.H * g.W * g.C;
  const bool dma_ok = aligned && data_bytes < (1LL << 31) &&
                      static_cast<long long>(O) * K < (1LL << 31);
  if (plan.cfg == 0) {
    const long cus = num_cus();
    auto tiles = [&](int bm, int bn) {
      return static_cast<long>((M + bm - 1) / bm) * ((O + bn - 1) / bn);
    };
    int auto_splits = 1;
    const bool may_split = force.splits != 1;
    if (dma_ok && few_tiles_wins(M, O, K, cus, may_split) &&
        few_tiles_conv_ok(g.C, K, g.KH, g.KW)) {
      plan.cfg = 63;
      plan.splits = 1;
      return plan;
    }
    if (dma_ok) {
      switch (choose_tile(M, O, K, cus, true, may_split ? &auto_splits : nullptr)) {
        case Tile::kL8: plan.cfg = 11; break;
        case Tile::kW128x2: plan.cfg = 22; break;
        case Tile::kW128K2: plan.cfg = 36; break;
        case Tile::kM128x2: plan.cfg = 24; break;
        case Tile::kM128K2: plan.cfg = 33; break;
        case Tile::kS64x2: plan.cfg = 25; break;
        case Tile::kS64K2: plan.cfg = 31; break;
        case Tile::kR128K2: plan.cfg = 37; break;
        case Tile::kQ128K2: plan.cfg = 38; break;
        case Tile::kS64K4: plan.cfg = 39; break;
        case Tile::kW64x2: plan.cfg = 23; break;
        case Tile::kS64S4: plan.cfg = 40; break;
        case Tile::kN32S3: plan.cfg = 41; break;
        case Tile::kN32K2: plan.cfg = 42; break;
        case Tile::kM128S3: plan.cfg = 43; break;
        case Tile::kW192K2:
          MXQ_CHECK(false, "a tile of plain operands proposed for gathered ones");
      }
    } else if (O > 128 && tiles(256, 256) >= cus) {
      plan.cfg = 1;
    } else if (O > 64 && tiles(256, 128) >= cus) {
      plan.cfg = 2;
    } else if (O <= 64 && tiles(256, 64) >= cus) {
      plan.cfg = 3;
    } else if (tiles(128, 128) >= cus) {
      plan.cfg = 4;
    } else {
      plan.cfg = 5;
    }
    if (plan.splits == 0) plan.splits = auto_splits;
  }
  if (plan.splits <= 0) plan.splits = 1;
  return plan;
}

// Channels that are no multiple of 16: copies of both operands with the channels padded, where
// the caller brought room for them (the loader of the register-staged kernels fetches such
// channels byte by byte: 21 x 29 x 29 x 17 -> 64, 7 x 7, 690 us against 14).
int conv_padded_c(const ConvGeometry& g) {
  const int Cp = (g.C + 15) / 16 * 16;
  const bool wanted = Cp != g.C && static_cast<long long>(g.N) * g.H * g.W * Cp < (1LL << 31) &&
                      static_cast<long long>(g.O) * g.KH * g.KW * Cp < (1LL << 31) &&
                      static_cast<long long>(g.N) * g.H * g.W * g.C >= 16 &&
                      static_cast<long long>(g.O) * g.K >= 16;
  return wanted ? Cp : 0;
}
size_t conv_padded_data(const ConvGeometry& g, int Cp) {
  return (static_cast<size_t>(g.N) * g.H * g.W * Cp + 255) / 256 * 256;
}
size_t conv_padded_bytes(const ConvGeometry& g, int Cp) {
  return conv_padded_data(g, Cp) +
         (static_cast<size_t>(g.O) * g.KH * g.KW * Cp + 255) / 256 * 256;
}

size_t conv_plan_workspace(const ConvPlan& plan, const ConvGeometry& g) {
  int bm, bn;
  if (plan.splits <= 1 || !conv_cfg_tile(plan.cfg, bm, bn)) return 0;
  const long tiles = static_cast<long>((g.M + bm - 1) / bm) * ((g.O + bn - 1) / bn);
  return splitk_workspace_bytes(tiles, plan.splits, bm, bn);
}

// ... with the workspace at hand: a split that the chooser proposed is dropped without room for it.
ConvPlan plan_conv_within(const ConvGeometry& g, bool aligned, const GemmForce& force,
                          const Workspace& ws) {
  const ConvPlan plan = plan_conv(g, aligned, force);
  if (force.splits != 0 || plan.splits <= 1 ||
      (ws.ptr != nullptr && aligned16(ws.ptr) && ws.bytes >= conv_plan_workspace(plan, g)))
    return plan;
  GemmForce unsplit = force;
  unsplit.splits = 1;
  return plan_conv(g, aligned, unsplit);
}

// Both C entry points: `planar` writes out32 as [N][O][OH][OW] instead of [N][OH][OW][O].
void conv_nhwc(void* stream, const int8_t* data, const int8_t* weight, const int8_t* bias, int N,
               int H, int W, int C, int O, int KH, int KW, int stride_h, int stride_w, int pad_h,
               int pad_w, int dilate_h, int dilate_w, const float* min_data,
               const float* max_data, const float* min_weight, const float* max_weight,
               const float* min_bias, const float* max_bias, int32_t* out32, float* omin,
               float* omax, int8_t* out8, float* rmin, float* rmax, int relu, float min_calib,
               float max_calib, bool planar, const GemmForce& force, const Workspace& ws,
               const void* prepared = nullptr) {
  const ConvGeometry g = conv_geometry(N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
                                       dilate_h, dilate_w);
  if (prepared == nullptr) {
    MXQ_CHECK(min_data && max_data && min_weight && max_weight, "null input range pointer");
    MXQ_CHECK(omin && omax, "null output range pointer");
    MXQ_CHECK(bias == nullptr || (min_bias && max_bias), "bias given without its range");
    MXQ_CHECK(out8 == nullptr || (rmin && rmax), "fused requantize needs rmin/rmax");
  }
  MXQ_CHECK(N == 0 || out32 != nullptr || out8 != nullptr, "no output buffer");
  ConvArgs a;
  a.data = data;
  a.weight = weight;
  a.N = N; a.H = H; a.W = W; a.C = C; a.O = O; a.KH = KH; a.KW = KW;
  a.sh = stride_h; a.sw = stride_w; a.ph = pad_h; a.pw = pad_w; a.dh = dilate_h; a.dw = dilate_w;
  a.OH = g.OH;
  a.OW = g.OW;
  a.M = static_cast<int>(g.M);
  a.K = static_cast<int>(g.K);
  a.sk.splits = 1;
  a.sk.kt_per_split = 1 << 30;
  a.sk.counters = nullptr;
  a.sk.partials = nullptr;
  MXQ_CHECK(a.M == 0 || O == 0 || (data != nullptr && weight != nullptr),
            "null operand pointer");
  Epilogue& e = a.epi;
  e.bias = bias;
  e.min_data = min_data; e.max_data = max_data;
  e.min_weight = min_weight; e.max_weight = max_weight;
  e.min_bias = min_bias; e.max_bias = max_bias;
  e.out32 = out32; e.out8 = out8; e.outf = nullptr;
  e.res = nullptr; e.res_min = nullptr; e.res_max = nullptr;
  e.sum_min_calib = 0.f; e.sum_max_calib = 0.f; e.sum_relu = 0; e.sum_requant = 0; e.with_sum = 0;
  e.sum_pairs = nullptr;
  e.prepared = static_cast<const char*>(prepared);
  e.omin = omin; e.omax = omax; e.rmin = rmin; e.rmax = rmax;
  e.relu = relu;
  float x = fabsf(min_calib), y = fabsf(max_calib);
  e.real_range = (x < y) ? y : x;
  e.plane = planar ? a.OH * a.OW : 0;
  e.stream8 = epi_stream_rows(a.M);

  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a.M == 0 || O == 0) {
    // no output elements: launch_fc writes the range scalars alone
    launch_fc(s, data, weight, a.M, O, C, O, e, GemmForce(), Workspace());
    return;
  }
  // a 1x1, unit-stride, unpadded convolution is the FC of the flattened pixels
  if (force.cfg == 0 && g.is_fc) {
    launch_fc(s, data, weight, a.M, O, C, O, e, force, ws);
    return;
  }
  if (const int Cp = force.cfg == 0 && C % 16 != 0 ? conv_padded_c(g) : 0) {
    const size_t copies = conv_padded_bytes(g, Cp);
    if (ws.ptr != nullptr && aligned16(ws.ptr) && ws.bytes >= copies) {
      int8_t* d = static_cast<int8_t*>(ws.ptr);
      int8_t* w = d + conv_padded_data(g, Cp);
      launch_pad_rows(s, data, static_cast<long long>(N) * H * W, d, weight,
                      static_cast<long long>(O) * KH * KW, w, C, Cp);
      Workspace rest;
      rest.ptr = d + copies;
      rest.bytes = ws.bytes - copies;
      conv_nhwc(stream, d, w, bias, N, H, W, Cp, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
                dilate_h, dilate_w, min_data, max_data, min_weight, max_weight, min_bias,
                max_bias, out32, omin, omax, out8, rmin, rmax, relu, min_calib, max_calib, planar,
                force, rest, prepared);
      return;
    }
  }
  const bool aligned = (C % 16 == 0) && aligned16(data) && aligned16(weight);
  const long long data_bytes = static_cast<long long>(N) * H * W * C;
  const bool dma_ok = aligned && data_bytes < (1LL << 31) &&
                      static_cast<long long>(O) * a.K < (1LL << 31);
  // 65: 1 x 1 layers with the weights in registers, where that is the faster way
  if ((force.cfg == 0 || force.cfg == 65) && KH == 1 && KW == 1 && pad_h == 0 && pad_w == 0) {
    ResidentArgs r = {};
    r.data = data;
    r.weight = weight;
    r.M = a.M;
    r.N = r.ldo = O;
    r.K = C;
    r.epi = e;
    r.area = a.OH * a.OW;
    r.OW = a.OW;
    r.image = static_cast<long long>(H) * W * C;
    r.down = stride_h * W * C;
    r.right = stride_w * C;
    r.images = N;
    if (resident_wins(r, aligned && aligned16(out8))) {
      launch_resident(s, r);
      return;
    }
  }
  MXQ_CHECK(force.cfg != 65, "not a layer for the kernel with the weights in registers");
  const ConvPlan plan = plan_conv_within(g, aligned, force, ws);
  // 61: the parked-weights row kernel (3 x 3 over 64 -> 64 channels, fused int8 output);
  // chosen for it whenever the launch has rows for every wave of the chip, with int32 planes by a
  // rule of their own
  const bool planes = a.epi.out32 != nullptr;
  if (plan.cfg == 61 ||
      (force.cfg == 0 && conv3x3_rows_ok(a) &&
       (planes ? conv3x3_rows_wins_planes(a)
               : static_cast<long>(a.N) * a.OH >= 1L * kRowsWaves * num_cus()))) {
    MXQ_CHECK(conv3x3_rows_ok(a), "shape does not qualify for the parked-weights 3x3 kernel");
    MXQ_CHECK(plan.splits <= 1 || force.splits == 0, "the 3x3 row kernel has no split-K form");
    launch_conv3x3_rows(s, a);
    return;
  }
  // 64: the few-tap kernel; chosen once two waves of every SIMD have an item (4 x 4 taps, 64
  // outputs: 25088 pixels 5.6 us tiled and 5.1 here, 12544 pixels 5.1 both)
  if (plan.cfg == 64 || (force.cfg == 0 && plan.splits <= 1 && conv_taps_ok(a) &&
                         a.M >= 64L * num_cus())) {
    MXQ_CHECK(conv_taps_ok(a), "shape does not qualify for the few-tap kernel");
    launch_conv_taps(s, a);
    return;
  }
  // 62: the resident-patch 3 x 3 kernel; chosen where it was measured ahead of the tiled
  // kernels (28 x 28 planes over 128 channels at batch 64: 15.4 against 16.6 us of kernel time)
  const long patch_tiles = static_cast<long>((a.M + 127) / 128) * ((a.O + 127) / 128);
  if (plan.cfg == 62 || (force.cfg == 0 && plan.splits <= 1 && conv3x3_patch_ok(a) &&
                         patch_tiles >= num_cus())) {
    MXQ_CHECK(conv3x3_patch_ok(a), "shape does not qualify for the resident-patch 3x3 kernel");
    MXQ_CHECK(plan.splits <= 1 || force.splits == 0, "the patch kernel has no split-K form");
    launch_conv3x3_patch(s, a);
    return;
  }
  // 66, 67: the window kernel on 128 and 256 pixels
  const int window = force.cfg == 66 || force.cfg == 67 ? force.cfg
                     : force.cfg == 0 && plan.cfg != 63 && dma_ok ? window_cfg(a) : 0;
  if (window != 0) {
    MXQ_CHECK(dma_ok && force.splits <= 1, "shape does not qualify for the window kernel");
    if (window == 66 ? launch_window<CfgWindow>(s, a) : launch_window<CfgWindow2>(s, a)) return;
    MXQ_CHECK(force.cfg == 0, "shape does not qualify for the window kernel");
  }
  const int cfg = plan.cfg, sp = plan.splits;
  if (cfg == 63) {  // the few-tiles kernel; `splits` is the number of waves per tile
    MXQ_CHECK(dma_ok && few_tiles_conv_ok(C, a.K, KH, KW),
              "shape does not qualify for the few-tiles kernel");
    FewTilesArgs f = {};
    f.data = data; f.weight = weight; f.M = a.M; f.N = O; f.K = a.K; f.ldo = O; f.epi = e;
    f.images = N; f.H = H; f.W = W; f.C = C; f.KW = KW; f.sh = a.sh; f.sw = a.sw; f.ph = a.ph;
    f.pw = a.pw; f.dh = a.dh; f.dw = a.dw; f.OH = a.OH; f.OW = a.OW;
    launch_few_tiles_conv(s, f,
                          force.splits != 0 ? force.splits : few_tiles_waves(a.M, O, a.K, true));
    return;
  }
  if (cfg > 10) MXQ_CHECK(dma_ok, "shape does not qualify for the direct-to-LDS conv kernels");
  if (cfg <= 10) MXQ_CHECK(sp <= 1, "the register-staged kernels have no split-K form");
  switch (cfg) {
    case 1: launch_cfg<CfgL8>(s, a, aligned); break;
    case 2: launch_cfg<CfgW128>(s, a, aligned); break;
    case 3: launch_cfg<CfgW64>(s, a, aligned); break;
    case 4: launch_cfg<CfgM>(s, a, aligned); break;
    case 5: launch_cfg<CfgS>(s, a, aligned); break;
    case 11: launch_dma<CfgL8, 4, 2>(s, a, sp, ws); break;
    case 31: launch_dma<CfgSK, 2, 0>(s, a, sp, ws); break;
    case 33: launch_dma<CfgMK, 2, 0>(s, a, sp, ws); break;
    case 36: launch_dma<CfgW128K, 2, 0>(s, a, sp, ws); break;
    case 37: launch_dma<CfgRK, 2, 0>(s, a, sp, ws); break;
    case 38: launch_dma<CfgQK, 2, 0>(s, a, sp, ws); break;
    case 39: launch_dma<CfgSK2, 2, 0>(s, a, sp, ws); break;
    case 40: launch_sliced<SlicedCfg<64, 64, 256>, 4>(s, a, sp, ws); break;
    case 41: launch_sliced<SlicedCfg<128, 32, 256>, 3>(s, a, sp, ws); break;
    case 43: launch_sliced<SlicedCfg<128, 128, 128>, 3>(s, a, sp, ws); break;
    case 42: launch_dma<CfgNK, 2, 0>(s, a, sp, ws); break;
    case 22: launch_dma<CfgW128, 2, 0>(s, a, sp, ws); break;
    case 23: launch_dma<CfgW64, 2, 0>(s, a, sp, ws); break;
    case 24: launch_dma<CfgM, 2, 0>(s, a, sp, ws); break;
    case 25: launch_dma<CfgS, 2, 0>(s, a, sp, ws); break;
#ifdef MXQ_TEST_HOOKS  // nothing proposes these
    case 12: launch_dma<CfgW128, 4, 2>(s, a, sp, ws); break;
    case 13: launch_dma<CfgW64, 4, 2>(s, a, sp, ws); break;
    case 14: launch_dma<CfgM, 4, 2>(s, a, sp, ws); break;
    case 15: launch_dma<CfgS, 4, 2>(s, a, sp, ws); break;
    case 16: launch_dma<CfgL4, 4, 2>(s, a, sp, ws); break;
    case 32: launch_dma<CfgSK, 3, 0>(s, a, sp, ws); break;
    case 34: launch_dma<CfgMK, 3, 0>(s, a, sp, ws); break;
    case 35: launch_dma<CfgL8K, 2, 0>(s, a, sp, ws); break;
#endif
    default: MXQ_CHECK(false, "unknown conv tile configuration " << cfg);
  }
}

}  // namespace

namespace {

struct PairLayer {
  const int8_t* weight;
  const void* prepared;
  int O;
  int8_t* out8;
  int relu;
  float min_calib, max_calib;
};

enum class PairRoute { kNone, kResident, kFewTiles, kTiles64, kTiles64Deep, kTiles128 };

// How two 1 x 1 convolutions of the same images go out as one launch, and whether that is faster
// than two.
PairRoute pair_route(const ConvGeometry& g, int O1, int O2) {
  const long long M = g.M, data = static_cast<long long>(g.N) * g.H * g.W * g.C;
  const int O = O1 + O2;
  if (g.M == 0 || O1 % 16 != 0 || O2 % 16 != 0 || g.C % 16 != 0 || data >= (1LL << 31) ||
      static_cast<long long>(O) * g.C >= (1LL << 31))
    return PairRoute::kNone;
  const long cus = num_cus();
  ResidentArgs a = {}, b;
  a.M = static_cast<int>(M);
  a.K = g.C;
  a.epi.out8 = reinterpret_cast<int8_t*>(16);  // only whether there is one counts
  a.area = g.OH * g.OW;
  a.OW = g.OW;
  a.image = static_cast<long long>(g.H) * g.W * g.C;
  b = a;
  a.N = a.ldo = O1;
  b.N = b.ldo = O2;
  if (resident_pair_wins(a, b, true)) return PairRoute::kResident;
  const long few = few_tiles_count(M, O1) + few_tiles_count(M, O2);
  if (g.C >= 256 && 4 * few <= 5 * cus && few_tiles_conv_ok(g.C, g.C, 1, 1))
    return PairRoute::kFewTiles;
  auto tiles = [&](long bm, long bn) {
    return (M + bm - 1) / bm * ((O1 + bn - 1) / bn + (O2 + bn - 1) / bn);
  };
  if (tiles(64, 64) <= 4 * cus) return g.C >= 1024 ? PairRoute::kTiles64Deep : PairRoute::kTiles64;
  if (g.C >= 1024 && tiles(128, 128) <= 2 * cus) return PairRoute::kTiles128;
  return PairRoute::kNone;
}

void conv_pair(void* stream, const int8_t* data, int N, int H, int W, int C, int stride_h,
               int stride_w, const PairLayer& x, const PairLayer& y) {
  MXQ_CHECK(x.prepared && aligned16(x.prepared) && y.prepared && aligned16(y.prepared),
            "null or unaligned pointer");
  const ConvGeometry g =
      conv_geometry(N, H, W, C, x.O, 1, 1, stride_h, stride_w, 0, 0, 1, 1);
  MXQ_CHECK(y.O > 0, "bad shape");
  MXQ_CHECK(g.M == 0 || (data && x.weight && y.weight), "null operand pointer");
  MXQ_CHECK(g.M == 0 || (x.out8 && y.out8), "no output buffer");
  const bool aligned = aligned16(data) && aligned16(x.weight) && aligned16(y.weight) &&
                       aligned16(x.out8) && aligned16(y.out8);
  const PairRoute route = aligned ? pair_route(g, x.O, y.O) : PairRoute::kNone;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto epilogue = [&](const PairLayer& l) {
    Epilogue e = {};
    e.out8 = l.out8;
    e.prepared = static_cast<const char*>(l.prepared);
    e.relu = l.relu;
    const float lo = fabsf(l.min_calib), hi = fabsf(l.max_calib);
    e.real_range = (lo < hi) ? hi : lo;
    e.stream8 = 0;  // the next launches read both: 608.8 us for a ResNet-50 at batch 64, 603.3 so
    return e;
  };
  const int M = static_cast<int>(g.M);
  if (route == PairRoute::kNone) {
    for (const PairLayer* l : {&x, &y})
      conv_nhwc(stream, data, l->weight, nullptr, N, H, W, C, l->O, 1, 1, stride_h, stride_w, 0, 0,
                1, 1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                nullptr, l->out8, nullptr, nullptr, l->relu, l->min_calib, l->max_calib, false,
                GemmForce(), Workspace(), l->prepared);
  } else if (route == PairRoute::kResident) {
    ResidentArgs r[2] = {};
    for (int i = 0; i < 2; ++i) {
      const PairLayer& l = i == 0 ? x : y;
      r[i].data = data;
      r[i].weight = l.weight;
      r[i].M = M;
      r[i].N = r[i].ldo = l.O;
      r[i].K = C;
      r[i].epi = epilogue(l);
      if (!g.is_fc) {
        r[i].area = g.OH * g.OW;
        r[i].OW = g.OW;
        r[i].image = static_cast<long long>(H) * W * C;
        r[i].down = stride_h * W * C;
        r[i].right = stride_w * C;
        r[i].images = N;
      }
    }
    launch_resident_pair(s, r[0], r[1]);
  } else if (route == PairRoute::kFewTiles) {
    FewTilesArgs f[2] = {};
    for (int i = 0; i < 2; ++i) {
      const PairLayer& l = i == 0 ? x : y;
      f[i].data = data; f[i].weight = l.weight; f[i].M = M; f[i].N = f[i].ldo = l.O; f[i].K = C;
      f[i].epi = epilogue(l);
      f[i].images = N; f[i].H = H; f[i].W = W; f[i].C = C; f[i].KW = 1;
      f[i].sh = stride_h; f[i].sw = stride_w; f[i].dh = f[i].dw = 1;
      f[i].OH = g.OH; f[i].OW = g.OW;
    }
    const int waves = few_tiles_waves(M, x.O + y.O, C, true);
    launch_few_tiles_pair(s, f[0], f[1], waves == 16 ? 8 : waves);
  } else {
    ConvArgs a[2] = {};
    for (int i = 0; i < 2; ++i) {
      const PairLayer& l = i == 0 ? x : y;
      a[i].data = data; a[i].weight = l.weight;
      a[i].N = N; a[i].H = H; a[i].W = W; a[i].C = C; a[i].O = l.O; a[i].KH = a[i].KW = 1;
      a[i].sh = stride_h; a[i].sw = stride_w; a[i].dh = a[i].dw = 1;
      a[i].OH = g.OH; a[i].OW = g.OW; a[i].M = M; a[i].K = C;
      a[i].epi = epilogue(l);
      a[i].sk.splits = 1;
      a[i].sk.kt_per_split = 1 << 30;
    }
    if (route == PairRoute::kTiles128) launch_pair<CfgMK>(s, a[0], a[1]);
    else if (route == PairRoute::kTiles64Deep) launch_pair<CfgSK2>(s, a[0], a[1]);
    else launch_pair<CfgS>(s, a[0], a[1]);
  }
}

}  // namespace

// Data [N][C][H][W] -> [N][H][W][Cp] and weights [O][C][KH][KW] -> [O][KH][KW][Cp] for the
// NCHW operator's adapter route, in one launch where the data's kernel can carry the weights.
void nchw_to_nhwc_pair(hipStream_t s, const int8_t* data, int8_t* d_out, int N, int C, int H,
                       int W, int Cp, const int8_t* weight, int8_t* w_out, int O, int KH, int KW) {
  MXQ_CHECK(static_cast<long long>(H) * W < (1LL << 31), "image too large");
  const int taps = KH * KW;
  GatherJob job = no_job();
  if (w_out != nullptr && gather_job_ok(w_out, O, taps, Cp))
    job = gather_job(weight, w_out, O, C, taps, Cp);
  const bool rides = job.blocks != 0;
  if (static_cast<long long>(N) * Cp * H * W != 0)
    launch_transpose<int8_t>(s, data, d_out, N, C, H * W, Cp, &job);
  if (w_out == nullptr) return;
  if (rides && job.blocks == 0) return;   // carried
  launch_transpose<int8_t>(s, weight, w_out, O, C, taps, Cp);
}

}  // namespace mxq

using namespace mxq;

extern "C" {

size_t mxq_quantized_conv_workspace(int N, int H, int W, int C, int O, int KH, int KW,
                                    int stride_h, int stride_w, int pad_h, int pad_w,
                                    int dilate_h, int dilate_w, int fused_int8_only) {
  try {
    const ConvGeometry g = conv_geometry(N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
                                         dilate_h, dilate_w);
    if (g.M == 0) return 0;
    if (g.is_fc)
      return fc_workspace_bytes(static_cast<int>(g.M), O, C, fused_int8_only != 0 && O % 16 == 0);
    if (const int Cp = C % 16 != 0 ? conv_padded_c(g) : 0)
      return conv_padded_bytes(g, Cp) +
             mxq_quantized_conv_workspace(N, H, W, Cp, O, KH, KW, stride_h, stride_w, pad_h,
                                          pad_w, dilate_h, dilate_w, fused_int8_only);
    return conv_plan_workspace(plan_conv(g, C % 16 == 0, GemmForce()), g);
  } catch (...) {
    return 0;
  }
}

int mxq_quantized_conv_nhwc_prepared(void* stream, const int8_t* data, const int8_t* weight,
                                     const void* prepared, int N, int H, int W, int C, int O,
                                     int KH, int KW, int stride_h, int stride_w, int pad_h,
                                     int pad_w, int dilate_h, int dilate_w, int8_t* out8, int relu,
                                     float min_calib, float max_calib, void* workspace,
                                     size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(prepared != nullptr && aligned16(prepared), "null or unaligned pointer");
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  conv_nhwc(stream, data, weight, nullptr, N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
            dilate_h, dilate_w, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
            nullptr, nullptr, out8, nullptr, nullptr, relu, min_calib, max_calib, false,
            GemmForce(), ws, prepared);
  MXQ_API_END();
}

int mxq_quantized_conv_pair_fits(int N, int H, int W, int C, int O1, int O2, int stride_h,
                                 int stride_w) {
  try {
    return pair_route(conv_geometry(N, H, W, C, O1, 1, 1, stride_h, stride_w, 0, 0, 1, 1), O1, O2) !=
           PairRoute::kNone;
  } catch (...) {
    return 0;
  }
}

int mxq_quantized_conv_pair_prepared(void* stream, const int8_t* data, int N, int H, int W, int C,
                                     int stride_h, int stride_w, const int8_t* weight1,
                                     const void* prepared1, int O1, int8_t* out1, int relu1,
                                     float min_calib1, float max_calib1, const int8_t* weight2,
                                     const void* prepared2, int O2, int8_t* out2, int relu2,
                                     float min_calib2, float max_calib2) {
  MXQ_API_BEGIN();
  conv_pair(stream, data, N, H, W, C, stride_h, stride_w,
            {weight1, prepared1, O1, out1, relu1, min_calib1, max_calib1},
            {weight2, prepared2, O2, out2, relu2, min_calib2, max_calib2});
  MXQ_API_END();
}

int mxq_quantized_conv_nhwc(void* stream, const int8_t* data, const int8_t* weight,
                            const int8_t* bias, int N, int H, int W, int C, int O, int KH,
                            int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                            int dilate_h, int dilate_w, const float* min_data,
                            const float* max_data, const float* min_weight,
                            const float* max_weight, const float* min_bias,
                            const float* max_bias, int32_t* out32, float* omin, float* omax,
                            int8_t* out8, float* rmin, float* rmax, int relu, float min_calib,
                            float max_calib, void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  conv_nhwc(stream, data, weight, bias, N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
            dilate_h, dilate_w, min_data, max_data, min_weight, max_weight, min_bias, max_bias,
            out32, omin, omax, out8, rmin, rmax, relu, min_calib, max_calib, false, GemmForce(),
            ws);
  MXQ_API_END();
}

#ifdef MXQ_TEST_HOOKS
// Test-only twin of mxq_quantized_conv_nhwc (declared in tests/mxq_test_hooks.h): the tile
// configuration and the split-K factor come as arguments (0 = let the launcher choose).
int mxq_test_quantized_conv_nhwc(void* stream, const int8_t* data, const int8_t* weight,
                                 const int8_t* bias, int N, int H, int W, int C, int O, int KH,
                                 int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                                 int dilate_h, int dilate_w, const float* min_data,
                                 const float* max_data, const float* min_weight,
                                 const float* max_weight, const float* min_bias,
                                 const float* max_bias, int32_t* out32, float* omin,
                                 float* omax, int8_t* out8, float* rmin, float* rmax, int relu,
                                 float min_calib, float max_calib, void* workspace,
                                 size_t workspace_bytes, int cfg, int splits) {
  MXQ_API_BEGIN();
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  GemmForce force;
  force.cfg = cfg;
  force.splits = splits;
  conv_nhwc(stream, data, weight, bias, N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
            dilate_h, dilate_w, min_data, max_data, min_weight, max_weight, min_bias, max_bias,
            out32, omin, omax, out8, rmin, rmax, relu, min_calib, max_calib, false, force, ws);
  MXQ_API_END();
}

// tests/mxq_test_hooks.h
int mxq_test_conv_plan(int N, int H, int W, int C, int O, int KH, int KW, int stride_h, int stride_w,
                       int pad_h, int pad_w, int dilate_h, int dilate_w, void* workspace,
                       size_t workspace_bytes, int* cfg, int* splits) {
  MXQ_API_BEGIN();
  MXQ_CHECK(C % 16 == 0 && cfg != nullptr && splits != nullptr, "whole pieces of channels");
  const ConvGeometry g = conv_geometry(N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
                                       dilate_h, dilate_w);
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  const ConvPlan plan = plan_conv_within(g, true, GemmForce(), ws);
  ConvArgs a = {};
  a.N = N; a.H = H; a.W = W; a.C = C; a.O = O; a.KH = KH; a.KW = KW;
  a.sh = stride_h; a.sw = stride_w; a.ph = pad_h; a.pw = pad_w; a.dh = dilate_h; a.dw = dilate_w;
  a.OH = g.OH; a.OW = g.OW;
  a.M = static_cast<int>(g.M);
  a.K = static_cast<int>(g.K);
  const int window = plan.cfg != 63 ? window_cfg(a) : 0;
  WindowArgs t;
  const bool fits = window == 66   ? window_layout<CfgWindow>(a, t) != 0
                    : window == 67 ? window_layout<CfgWindow2>(a, t) != 0 : false;
  *cfg = fits ? window : plan.cfg;
  *splits = fits ? 1 : plan.splits;
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

int mxq_quantized_conv_nhwc_out_nchw(void* stream, const int8_t* data, const int8_t* weight,
                                     const int8_t* bias, int N, int H, int W, int C, int O,
                                     int KH, int KW, int stride_h, int stride_w, int pad_h,
                                     int pad_w, int dilate_h, int dilate_w,
                                     const float* min_data, const float* max_data,
                                     const float* min_weight, const float* max_weight,
                                     const float* min_bias, const float* max_bias,
                                     int32_t* out32_nchw, float* omin, float* omax,
                                     void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(out32_nchw != nullptr, "no output buffer");
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  conv_nhwc(stream, data, weight, bias, N, H, W, C, O, KH, KW, stride_h, stride_w, pad_h, pad_w,
            dilate_h, dilate_w, min_data, max_data, min_weight, max_weight, min_bias, max_bias,
            out32_nchw, omin, omax, nullptr, nullptr, nullptr, 0, 0.f, 0.f, true, GemmForce(), ws);
  MXQ_API_END();
}


int mxq_nchw_to_nhwc_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                        int W) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && C >= 0 && H >= 0 && W >= 0, "negative dimension");
  MXQ_CHECK((static_cast<long long>(H) * W) < (1LL << 31), "image too large");
  if (static_cast<long long>(N) * C * H * W == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  launch_transpose<int8_t>(static_cast<hipStream_t>(stream), in, out, N, C, H * W, C);
  MXQ_API_END();
}

int mxq_nchw_to_nhwc_pad_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int C_padded) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && C >= 0 && H >= 0 && W >= 0, "negative dimension");
  MXQ_CHECK(C_padded >= C, "C_padded must be at least C");
  MXQ_CHECK((static_cast<long long>(H) * W) < (1LL << 31), "image too large");
  if (static_cast<long long>(N) * C_padded * H * W == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  launch_transpose<int8_t>(static_cast<hipStream_t>(stream), in, out, N, C, H * W, C_padded);
  MXQ_API_END();
}

int mxq_nchw_to_s2d_nhwc_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int off_h, int off_w, int C_padded) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && C >= 0 && H >= 0 && W >= 0, "negative dimension");
  MXQ_CHECK((off_h == 0 || off_h == 1) && (off_w == 0 || off_w == 1), "offsets are 0 or 1");
  MXQ_CHECK(C_padded >= 4 * C, "C_padded must be at least 4 * C");
  const int H2 = (H + off_h + 1) / 2, W2 = (W + off_w + 1) / 2;
  const size_t pixels = static_cast<size_t>(N) * H2 * W2;
  if (pixels == 0 || C_padded == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  size_t g = (pixels + 255) / 256;
  if (g > 65535u * 16u) g = 65535u * 16u;
  hipLaunchKernelGGL(s2d_nhwc_kernel, dim3(static_cast<unsigned>(g)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), in, out, C, H, W, H2, W2, off_h, off_w,
                     C_padded, pixels);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_nhwc_to_nchw(void* stream, const void* in, void* out, int N, int C, int H, int W,
                     int elem_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0 && C >= 0 && H >= 0 && W >= 0, "negative dimension");
  MXQ_CHECK(elem_bytes == 1 || elem_bytes == 4, "elem_bytes must be 1 or 4");
  MXQ_CHECK((static_cast<long long>(H) * W) < (1LL << 31), "image too large");
  if (static_cast<long long>(N) * C * H * W == 0) return 0;
  MXQ_CHECK(in != nullptr && out != nullptr, "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (elem_bytes == 1)
    launch_transpose<int8_t>(s, in, out, N, H * W, C, H * W);
  else
    launch_transpose<int32_t>(s, in, out, N, H * W, C, H * W);
  MXQ_API_END();
}

}  // extern "C"
