// The fully-connected kernels and their launch templates (see mxq_fc.hip for the operator
// they serve and the list of tile configurations).  Included by one translation unit per
// epilogue mode, which instantiates every configuration for that mode through
// fc_launch_mode<MODE>.
#ifndef MXQ_FC_KERNELS_H_
#define MXQ_FC_KERNELS_H_

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_fc_args.h"
#include "mxq_gemm.h"
#include "mxq_tiles.h"

namespace mxq {

namespace {


template <class Cfg, bool ALIGNED, int MODE>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kMinWaves) void fc_kernel(FcArgs p) {
  __shared__ __attribute__((aligned(16))) v4i lds[2][Cfg::STAGE_SLOTS];
  const int wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;

  RowFetch<Cfg, Cfg::A_CHUNKS, ALIGNED> af;
  RowFetch<Cfg, Cfg::B_CHUNKS, ALIGNED> bf;
  af.init(p.data, m0, p.M, p.K);
  bf.init(p.weight, n0, p.N, p.K);

  v16i acc[Cfg::MI][Cfg::NI];
  gemm_mainloop<Cfg>(acc, af, bf, (p.K + Cfg::BK - 1) / Cfg::BK, lds);

  gemm_epilogue<Cfg, MODE>(acc, p.epi, m0 + wm * Cfg::TM, n0 + wn * Cfg::TN, p.M, p.N,
                     static_cast<size_t>(p.ldo));
  if (blockIdx.x == 0 && threadIdx.x == 0) epilogue_ranges<MODE>(p.epi);
}

// Direct-to-LDS variant (see gemm_mainloop_dma); launch_fc() picks it when the
// operands qualify.  BUF selects buffer loads (any K % 16 == 0, zero-filled tails)
// over global loads (K % 64 == 0, clamped rows).
// MODE (kEpiPlain / kEpiF32 / kEpiSum) builds the float output or the residual sum in: kernels
// of their own, so that the int8 and int32 forms do not carry their code.
template <class Cfg, int NS, int PIPE, bool BUF, int MODE>
__global__ __launch_bounds__(Cfg::kThreads, NS <= 2 ? Cfg::kMinWaves : 1) void fc_dma_kernel(FcArgs p) {
  __shared__ __attribute__((aligned(16))) v4i lds[NS * Cfg::STAGE_SLOTS];
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn, tile = 0, z = 0;
  if (__builtin_expect(p.sk.splits > 1, 0))
    tile_coords_split(blockIdx.x, tiles_m, tiles_n, p.sk.splits, tm, tn, tile, z);
  else
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // what the epilogue needs is fetched while the first operand stages are in flight
  EpiPreOf<MODE> pre;
  auto prefetch = [&]() { pre = epi_prefetch<Cfg, MODE>(p.epi, n0, p.N); };
  v16i acc[Cfg::MI][Cfg::NI];
  // this work-group's K slice: stages [kt0, kt0 + KT) (all of them without a split)
  const int kt_all = (p.K + Cfg::BK - 1) / Cfg::BK;
  const int kt0 = z * p.sk.kt_per_split;
  const int KT = (kt_all - kt0) < p.sk.kt_per_split ? (kt_all - kt0) : p.sk.kt_per_split;
  const int kbeg = kt0 * Cfg::BK;
  if (BUF) {
    RowIssuerBuffer<Cfg, Cfg::A_CHUNKS> ai;
    RowIssuerBuffer<Cfg, Cfg::B_CHUNKS> bi;
    ai.init(p.data, m0, p.M, p.K, wave, lane, kbeg);
    bi.init(p.weight, n0, p.N, p.K, wave, lane, kbeg);
    gemm_mainloop_dma<Cfg, NS, PIPE>(acc, ai, bi, KT, lds, prefetch);
  } else {
    RowIssuerGlobal<Cfg, Cfg::A_CHUNKS> ai;
    RowIssuerGlobal<Cfg, Cfg::B_CHUNKS> bi;
    ai.init(p.data, m0, p.M, p.K, wave, lane, kbeg);
    bi.init(p.weight, n0, p.N, p.K, wave, lane, kbeg);
    gemm_mainloop_dma<Cfg, NS, PIPE>(acc, ai, bi, KT, lds, prefetch);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (blockIdx.x == 0 && threadIdx.x == 0) epilogue_ranges<MODE>(p.epi);
  if (__builtin_expect(p.sk.splits > 1, 0) && !splitk_gather<Cfg>(acc, p.sk, tile, z)) return;

  gemm_epilogue_lds<Cfg, NS * Cfg::STAGE_SLOTS * 16, MODE>(acc, p.epi, pre, m0, n0, p.M, p.N,
                                                           static_cast<size_t>(p.ldo), lds);
}

// A tile on eight waves (gemm_mainloop_sliced).
template <class Cfg, int NS, int MODE>
__global__ __launch_bounds__(Cfg::kThreads, 2) void fc_sliced_kernel(FcArgs p) {
  typedef typename Cfg::Tile Tile;
  __shared__ __attribute__((aligned(16))) v4i lds[NS * Cfg::STAGE_SLOTS];
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn, tile = 0, z = 0;
  if (__builtin_expect(p.sk.splits > 1, 0))
    tile_coords_split(blockIdx.x, tiles_m, tiles_n, p.sk.splits, tm, tn, tile, z);
  else
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  EpiPreOf<MODE> pre;
  auto prefetch = [&]() { pre = epi_prefetch<Tile, MODE>(p.epi, n0, p.N); };
  const int kt_all = (p.K + Cfg::BK - 1) / Cfg::BK;
  const int kt0 = z * p.sk.kt_per_split;
  const int KT = (kt_all - kt0) < p.sk.kt_per_split ? (kt_all - kt0) : p.sk.kt_per_split;
  RowIssuerBuffer<Cfg, Cfg::A_CHUNKS> ai;
  RowIssuerBuffer<Cfg, Cfg::B_CHUNKS> bi;
  ai.init(p.data, m0, p.M, p.K, wave, lane, kt0 * Cfg::BK);
  bi.init(p.weight, n0, p.N, p.K, wave, lane, kt0 * Cfg::BK);
  if (blockIdx.x == 0 && threadIdx.x == 0) epilogue_ranges<MODE>(p.epi);
  v16i acc[1][Cfg::NI];
  if (!gemm_mainloop_sliced<Cfg, NS>(acc, ai, bi, KT, lds, prefetch)) return;
  if (__builtin_expect(p.sk.splits > 1, 0) && !splitk_gather<Tile>(acc, p.sk, tile, z)) return;
  gemm_epilogue_lds<Tile, NS * Cfg::STAGE_SLOTS * 16, MODE>(acc, p.epi, pre, m0, n0, p.M, p.N,
                                                            static_cast<size_t>(p.ldo), lds);
}

typedef GemmCfg<256, 256, 64, 2, 4> CfgL8;    // 8 waves, wave tile 128 x 64
typedef GemmCfg<256, 256, 64, 2, 2> CfgL4;    // 4 waves, wave tile 128 x 128
typedef GemmCfg<256, 128, 64, 4, 2> CfgW128;  // 8 waves, wave tile 64 x 64
typedef GemmCfg<256, 64, 64, 4, 1> CfgW64;    // 4 waves, wave tile 64 x 64
typedef GemmCfg<128, 128, 64, 2, 2> CfgM;     // 4 waves, wave tile 64 x 64
typedef GemmCfg<64, 64, 64, 2, 2> CfgS;       // 4 waves, wave tile 32 x 32
// 128-byte stages: half as many K steps (each costs a barrier and a round of DMA latency)
typedef GemmCfg<256, 256, 128, 2, 4> CfgL8K;   // 8 waves, wave tile 128 x 64
typedef GemmCfg<256, 128, 128, 4, 2> CfgW128K; // 8 waves, wave tile 64 x 64
typedef GemmCfg<128, 128, 128, 2, 2> CfgMK;    // 4 waves, wave tile 64 x 64
typedef GemmCfg<64, 64, 128, 2, 2> CfgSK;      // 4 waves, wave tile 32 x 32
typedef GemmCfg<128, 64, 128, 2, 2> CfgRK;     // 4 waves, wave tile 64 x 32
typedef GemmCfg<64, 128, 128, 2, 2> CfgQK;     // 4 waves, wave tile 32 x 64
typedef GemmCfg<64, 64, 256, 2, 2> CfgSK2;     // 256-byte stages for very long K
typedef GemmCfg<256, 192, 128, 4, 2> CfgW192K; // 8 waves, wave tile 64 x 96

// Short-K form (K = 32, 64, 128 or 256; int8 output only).  With one or two K steps a tile of
// the kernels above is all prologue and epilogue: a round of DMA latency, two barriers, and
// an epilogue that keeps the CU's VALUs busy half the time.  Here the weight strip of a
// work-group (up to 256 rows of K bytes, 128 for K = 256) is parked in LDS once, and every wave on its own
// streams work items "32 data rows x 32*NI columns": the data fragment straight from global
// memory into the MFMA layout (a row of K bytes is consumed whole by the wave's K/16 loads),
// the next item's fragment requested before the current one is multiplied, weights read from
// LDS, then the fused epilogue and a transpose of the int8 tile through the wave's own LDS
// scratch.  No barrier after the weights are staged; waves only meet the memory system.
// A sum MODE: the residual operand FcArgs::epi.res is added to the int8 tile on its way out.
constexpr int kNonTemporal = 2;  // the buffer instructions' nt bit
__device__ __forceinline__ __amdgpu_buffer_rsrc_t stream_rsrc(const int8_t* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p), 0, bytes, 0x00020000);
}

template <int KS, int NI, int MODE>
__global__ __launch_bounds__(256, 2) void fc_stream_kernel(FcArgs p, int bn, int strips) {
  constexpr bool SUM = epi_sums(MODE);
  constexpr int K = 32 * KS, CH = 2 * KS;  // bytes and 16-byte chunks per row
  constexpr int TN = 32 * NI, LD = TN + 16;
  constexpr int LPR = TN / 16, RPI = 64 / LPR;
  constexpr int kMaxRows = KS <= 4 ? 256 : 128;  // weight rows per work-group: at most 32 KB
  __shared__ __attribute__((aligned(16))) v4i ldsB[kMaxRows * CH];
  __shared__ __attribute__((aligned(16))) int sbias[256];
  __shared__ __attribute__((aligned(16))) char stage_all[4 * 32 * LD];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_begin = blockIdx.y * bn;
  const int cols = (p.N - n_begin) < bn ? (p.N - n_begin) : bn;  // a multiple of TN
  for (int i = tid; i < cols * CH; i += 256) {
    const int r = i / CH, c = i - r * CH;
    ldsB[r * CH + (c ^ swz<CH>(r))] = *reinterpret_cast<const v4i*>(
        p.weight + static_cast<size_t>(n_begin + r) * K + c * 16);
  }
  const EpiScalars s = epi_scalars(p.epi);
  EpiPreOf<SUM ? MODE : kEpiSum> rules;
  if constexpr (SUM)
    rules.sum = epi_sum_rule<MODE>(p.epi);
  else
    rules.sum = SumRule{0.0f, 0.0f, 1};
  const auto& rule = rules.sum;
  if (tid < cols) sbias[tid] = epi_bias32(p.epi, s, n_begin + tid);
  __syncthreads();

  const int lrow = lane & 31, lgrp = lane >> 5;
  char* stage = stage_all + wave * 32 * LD;
  const int tiles_m = (p.M + 31) / 32;
  const int items = tiles_m * strips;
  const int step = gridDim.x * 4;
  // Both streams of an item come through a buffer descriptor of its own: what lies past the last
  // row, or past the last item (the loads of the last turn), arrives as zeros without being
  // fetched.  No branch around a load and nothing that looks at one before the next turn: with
  // either the compiler makes every turn wait for its own prefetch, and memory and arithmetic
  // take turns (200704 x 64 -> 256, one launch repeated over the same operands: 20.4 us, 17.2 now
  // at 3.7 TB/s; with the requantized sum 37.7, 28.2 now, 4.1 TB/s, the VALU busy for two thirds of
  // it.  Inside a network's pass the sum takes 28.8 to 30.5).
  constexpr int kRes = SUM ? 32 / RPI : 1;
  struct Item {
    v4i a[KS];
    v4i res[kRes];  // the residual operand's pieces, in the layout the tile leaves in
  };
  auto load = [&](int item, Item& f) {
    const int tile = item / strips;
    const int rows = item < items ? (p.M - tile * 32 < 32 ? p.M - tile * 32 : 32) : 0;
    const int first = rows > 0 ? tile * 32 : 0;
    const auto a = stream_rsrc(p.data + static_cast<size_t>(first) * K, rows * K);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      f.a[ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                            a, lrow * K + lgrp * 16 + ks * 32, 0, 0));
    if constexpr (SUM) {
      const auto r = stream_rsrc(p.epi.res + static_cast<size_t>(first) * p.ldo, rows * p.ldo);
      const int col = n_begin + (item - tile * strips) * TN + (lane % LPR) * 16;
#pragma unroll
      for (int it = 0; it < kRes; ++it)
        f.res[it] = __builtin_bit_cast(
            v4i, __builtin_amdgcn_raw_buffer_load_b128(
                     r, (it * RPI + lane / LPR) * p.ldo + col, 0, kNonTemporal));
    }
  };
  // One item: the next one's loads go out, this one is multiplied, finished and stored.
  // SM: 0 no sum, 1 sum, 2 sum + relu, 3 sum + relu in its short form, 4 / 5 as 1 / 2 where the
  // products could overflow
  auto turn = [&](int item, const Item& now, Item& next, auto stream, auto sum_mode,
                  auto with_relu) {
    constexpr int SM = decltype(sum_mode)::value;
    load(item + step, next);
    const int tile = item / strips;
    const int s0 = (item - tile * strips) * TN;  // first column of the strip inside the group's
    const int m_base = tile * 32;
    // the accumulators start at the int32 bias of their columns (read from LDS straight
    // into the registers the MFMAs add to): the epilogue has no bias add left
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
      for (int ni = 0; ni < NI; ++ni) {
        const int r = s0 + ni * 32 + lrow;
        const v4i fb = ldsB[r * CH + ((ks * 2 + lgrp) ^ swz<CH>(r))];
        acc[ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, now.a[ks], acc[ni], 0, 0, 0);
      }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int nl = ni * 32 + 8 * vq + 4 * lgrp;
        *reinterpret_cast<uint32_t*>(stage + lrow * LD + nl) =
            epi_requant_pack<decltype(with_relu)::value>(acc[ni][4 * vq], acc[ni][4 * vq + 1],
                                                         acc[ni][4 * vq + 2],
                                                         acc[ni][4 * vq + 3], s);
      }
    // the wave reads back what its own lanes wrote: LDS executes a wave's instructions in
    // order, the wait makes the writes complete first
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int rows = p.M - m_base < 32 ? p.M - m_base : 32;
    const auto out = stream_rsrc(p.epi.out8 + static_cast<size_t>(m_base) * p.ldo, rows * p.ldo);
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it) {
      const int rr = it * RPI + lane / LPR, c16 = lane % LPR;
      v4i val = *reinterpret_cast<const v4i*>(stage + rr * LD + c16 * 16);
      if constexpr (SM != 0) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          constexpr bool kRelu = SM == 2 || SM == 5, kFast = SM < 4;
          const uint32_t x = static_cast<uint32_t>(val[w]);
          const uint32_t y = static_cast<uint32_t>(now.res[it][w]);
          if constexpr (SM == 3)
            val[w] = static_cast<int>(epi_sum_pairs4(x, y, rules));
          else if constexpr (MODE == kEpiSumRq)
            val[w] = static_cast<int>(kFast ? sum_requant4<kRelu>(x, y, rule)
                                            : sum_requant4_general<kRelu>(x, y, rule));
          else
            val[w] = static_cast<int>(sum4<kRelu, kFast>(x, y, rule));
        }
      }
      __builtin_amdgcn_raw_buffer_store_b128(val, out, rr * p.ldo + n_begin + s0 + c16 * 16, 0,
                                             decltype(stream)::value ? kNonTemporal : kDeviceScope);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  };
  // Two items change places instead of registers being copied: a copy would wait for its loads,
  // and for the stores in front of them.
  auto run = [&](auto stream, auto sum_mode, auto with_relu) {
    int item = blockIdx.x * 4 + wave;
    Item x, y;
    load(item, x);
    while (item < items) {
      turn(item, x, y, stream, sum_mode, with_relu);
      item += step;
      if (item >= items) break;
      turn(item, y, x, stream, sum_mode, with_relu);
      item += step;
    }
  };
  auto run_flavour = [&](auto stream) {
    typedef std::false_type No;
    if constexpr (!SUM) {
      if (p.epi.relu)
        run(stream, std::integral_constant<int, 0>(), std::true_type());
      else
        run(stream, std::integral_constant<int, 0>(), No());
    } else {  // a layer in front of a sum has no relu of its own
      if (MODE == kEpiSumRq && epi_sum_pairs(rules))
        run(stream, std::integral_constant<int, MODE == kEpiSumRq ? 3 : 2>(), No());
      else if (rule.fast && p.epi.sum_relu)
        run(stream, std::integral_constant<int, 2>(), No());
      else if (rule.fast)
        run(stream, std::integral_constant<int, 1>(), No());
      else if (p.epi.sum_relu)
        run(stream, std::integral_constant<int, 5>(), No());
      else
        run(stream, std::integral_constant<int, 4>(), No());
    }
  };
  if (p.epi.stream8)
    run_flavour(std::true_type());
  else
    run_flavour(std::false_type());
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) epilogue_ranges<MODE>(p.epi);
}

template <int KS, int NI, int MODE>
void launch_stream(hipStream_t s, const FcArgs& a, long cus, int groups_per_cu) {
  // the residual operand is read in 16-byte pieces, like the output is written
  MXQ_CHECK(a.epi.res == nullptr || aligned16(a.epi.res), "unaligned residual operand");
  // 32 rows of the output are addressed with 32-bit byte offsets
  MXQ_CHECK(a.ldo < (1 << 25), "row pitch too large for the short-K streaming kernel");
  constexpr int TN = 32 * NI;
  const int max_rows = KS <= 4 ? 256 : 128;
  const int bn = a.N < max_rows ? a.N : max_rows;
  const int ny = (a.N + bn - 1) / bn;
  const int strips = bn / TN;
  const long items = static_cast<long>((a.M + 31) / 32) * strips;
  long gx = cus * groups_per_cu / ny;
  if (gx < 1) gx = 1;
  if (gx * 4 > items) gx = (items + 3) / 4;
  hipLaunchKernelGGL((fc_stream_kernel<KS, NI, MODE>), dim3(static_cast<unsigned>(gx), ny),
                     dim3(256), 0, s, a, bn, strips);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg, int NS, int PIPE, bool BUF, int MODE>
void launch_dma(hipStream_t s, FcArgs a, int splits, const Workspace& ws) {
  const long tiles = static_cast<long>((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.N + Cfg::BN - 1) / Cfg::BN);
  splitk_setup<Cfg>(s, a.sk, tiles, a.K, splits, ws.ptr, ws.bytes);
  hipLaunchKernelGGL((fc_dma_kernel<Cfg, NS, PIPE, BUF, MODE>),
                     dim3(static_cast<unsigned>(tiles * a.sk.splits)), dim3(Cfg::kThreads), 0, s,
                     a);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg, int NS, int MODE>
void launch_sliced(hipStream_t s, FcArgs a, int splits, const Workspace& ws) {
  const long tiles = static_cast<long>((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.N + Cfg::BN - 1) / Cfg::BN);
  splitk_setup<typename Cfg::Tile>(s, a.sk, tiles, a.K, splits, ws.ptr, ws.bytes);
  hipLaunchKernelGGL((fc_sliced_kernel<Cfg, NS, MODE>),
                     dim3(static_cast<unsigned>(tiles * a.sk.splits)), dim3(Cfg::kThreads), 0, s,
                     a);
  MXQ_LAUNCH_CHECK();
}

template <class Cfg, int MODE>
void launch_cfg(hipStream_t s, const FcArgs& a, bool aligned) {
  const int tiles = ((a.M + Cfg::BM - 1) / Cfg::BM) * ((a.N + Cfg::BN - 1) / Cfg::BN);
  if (aligned)
    hipLaunchKernelGGL((fc_kernel<Cfg, true, MODE>), dim3(tiles), dim3(Cfg::kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((fc_kernel<Cfg, false, MODE>), dim3(tiles), dim3(Cfg::kThreads), 0, s, a);
  MXQ_LAUNCH_CHECK();
}

// Every configuration for one epilogue mode.
template <int MODE>
void fc_launch_mode(hipStream_t s, const FcArgs& a, const FcLaunch& how, const Workspace& ws) {
  const int cfg = how.cfg, sp = how.splits;
  if (cfg == 61 || cfg == 62) {
    // the streaming kernel writes the int8 output (with or without the residual sum)
    if constexpr (MODE == kEpiF32) {
      MXQ_CHECK(false, "the short-K streaming kernel has no float-output form");
    } else {
      const long cus = num_cus();
#define MXQ_STREAM(NI)                                                             \
  do {                                                                             \
    if (a.K == 32) launch_stream<1, NI, MODE>(s, a, cus, how.stream_groups);        \
    else if (a.K == 64) launch_stream<2, NI, MODE>(s, a, cus, how.stream_groups);   \
    else if (a.K == 128) launch_stream<4, NI, MODE>(s, a, cus, how.stream_groups);  \
    else launch_stream<8, NI, MODE>(s, a, cus, how.stream_groups);                  \
  } while (0)
      if (cfg == 61) MXQ_STREAM(2); else MXQ_STREAM(4);
#undef MXQ_STREAM
    }
    return;
  }
  switch (cfg) {
    case 1: launch_cfg<CfgL8, MODE>(s, a, how.aligned); break;
    case 3: launch_cfg<CfgM, MODE>(s, a, how.aligned); break;
    case 4: launch_cfg<CfgS, MODE>(s, a, how.aligned); break;
    case 12: launch_dma<CfgL8, 4, 2, false, MODE>(s, a, sp, ws); break;
    case 41: launch_dma<CfgW128, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 43: launch_dma<CfgM, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 44: launch_dma<CfgS, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 51: launch_dma<CfgSK, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 53: launch_dma<CfgMK, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 55: launch_dma<CfgL8K, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 57: launch_dma<CfgRK, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 58: launch_dma<CfgQK, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 59: launch_dma<CfgSK2, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 60: launch_dma<CfgW192K, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 33: launch_sliced<SlicedCfg<64, 64, 256>, 4, MODE>(s, a, sp, ws); break;
    case 34: launch_sliced<SlicedCfg<128, 128, 128>, 3, MODE>(s, a, sp, ws); break;
    case 31: launch_dma<CfgL8, 4, 2, true, MODE>(s, a, sp, ws); break;
#ifdef MXQ_TEST_HOOKS  // nothing proposes these
    case 2: launch_cfg<CfgL4, MODE>(s, a, how.aligned); break;
    case 11: launch_dma<CfgL8, 4, 0, false, MODE>(s, a, sp, ws); break;
    case 14: launch_dma<CfgL4, 4, 0, false, MODE>(s, a, sp, ws); break;
    case 16: launch_dma<CfgL4, 4, 2, false, MODE>(s, a, sp, ws); break;
    case 21: launch_dma<CfgW128, 4, 2, true, MODE>(s, a, sp, ws); break;
    case 22: launch_dma<CfgW64, 4, 2, true, MODE>(s, a, sp, ws); break;
    case 23: launch_dma<CfgM, 4, 2, true, MODE>(s, a, sp, ws); break;
    case 24: launch_dma<CfgS, 4, 2, true, MODE>(s, a, sp, ws); break;
    case 42: launch_dma<CfgW64, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 52: launch_dma<CfgSK, 3, 0, true, MODE>(s, a, sp, ws); break;
    case 54: launch_dma<CfgMK, 3, 0, true, MODE>(s, a, sp, ws); break;
    case 56: launch_dma<CfgW128K, 2, 0, true, MODE>(s, a, sp, ws); break;
    case 32: launch_dma<CfgL4, 4, 2, true, MODE>(s, a, sp, ws); break;
#endif
    default: MXQ_CHECK(false, "unknown fc tile configuration " << cfg);
  }
}

}  // namespace

}  // namespace mxq
#endif  // MXQ_FC_KERNELS_H_
