// _contrib_quantized_fully_connected on gfx950: int8 data [M,K] x int8 weight
// [N,K]^T -> int32, with the int8 bias rescaled to int32 and (optionally) the
// calibrated requantize fused into the epilogue.  Replaces cublasGemmEx +
// QuantizedBiasAddKernel of the reference's GPU operator
// (src/operator/quantization/quantized_fully_connected.cu:58-138) with the exact
// integer semantics of its CPU operator (quantized_fully_connected.cc:149-297).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_fc_args.h"
#include "mxq_few_tiles.h"
#include "mxq_forms.h"
#include "mxq_resident.h"
#include "mxq_gemm.h"
#include "mxq_tiles.h"

namespace mxq {

// Tile configurations:
//   1..4    register-staged kernels (any shape): 256x256x8w, 256x256x4w, 128x128, 64x64
//   11, 12  direct-to-LDS 256x256, 8 waves: compiler-scheduled / pinned pipeline
//   14, 16  direct-to-LDS 256x256, 4 waves: compiler-scheduled / pinned pipeline
//   21..24  direct-to-LDS buffer-load kernels 256x128, 256x64, 128x128, 64x64
//   31, 32  as 12 / 16 with buffer loads (K % 16 == 0 instead of K % 64 == 0)
//   33, 34  64x64 and 128x128 on eight waves
//   41..44  as 21..24 with a 2-stage ring (short K)
//   51..56  128-byte stages: 64x64 (2, 3 stages), 128x128 (2, 3), 256x256 (2), 256x128 (2)
//   57..59  128x64 and 64x128 with 128-byte stages, 64x64 with 256-byte stages
//   60      256x192 with 128-byte stages (outputs whose width is a multiple of 192)
//   61, 62  the short-K streaming kernel with 64- / 128-column strips
//   65      the kernel with the weights in registers, where it is the faster one
//   71      the few-tiles kernel (any shape; here `splits` is the number of waves per
//           32 x 32 tile, negative for 16 x 16 tiles)
// plan_fc proposes 1, 3, 4, 12, 31, 33, 34, 41, 43, 44, 51, 53, 57..62 and 71, and 55 for a residual sum;
// the others are built with the test entries alone, for the tests that pin them.
// Output tile of a direct-to-LDS configuration (what a split-K work-group leaves in the
// workspace); false for every other configuration.
bool fc_cfg_tile(int cfg, int& bm, int& bn) {
  switch (cfg) {
    case 11: case 12: case 14: case 16: case 31: case 32: case 55: bm = 256; bn = 256; return true;
    case 21: case 41: case 56: bm = 256; bn = 128; return true;
    case 22: case 42: bm = 256; bn = 64; return true;
    case 23: case 43: case 53: case 54: case 34: bm = 128; bn = 128; return true;
    case 24: case 44: case 51: case 52: case 59: case 33: bm = 64; bn = 64; return true;
    case 57: bm = 128; bn = 64; return true;
    case 58: bm = 64; bn = 128; return true;
    case 60: bm = 256; bn = 192; return true;
    default: return false;
  }
}

struct FcPlan {
  int cfg;
  int splits;
  int stream_groups;
};

// What launch_fc would run for this shape.  `aligned`: K % 16 == 0 and 16-byte aligned
// operands; `fused8`: int8 output only, 16-byte aligned with a row pitch that is a
// multiple of 16 (what the streaming kernel stores).
// `sum`: the residual-sum form, whose epilogue does twice the arithmetic per output.
FcPlan plan_fc(int M, int N, int K, bool aligned, bool fused8, const GemmForce& force,
               bool sum = false,
               bool requant = false) {
  FcPlan plan = {force.cfg, force.splits, force.stream_groups > 0 ? force.stream_groups : 2};
  const bool buf_ok = aligned && K >= 16 && static_cast<long long>(M) * K < (1LL << 31) &&
                      static_cast<long long>(N) * K < (1LL << 31);
  const bool glb_ok = buf_ok && (K % 64 == 0);
  const long cus = num_cus();
  if (plan.cfg == 0) {
    auto tiles = [&](int bm, int bn) {
      return static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    };
    int auto_splits = 1;
    const bool may_split = force.splits != 1;
    if ((buf_ok && few_tiles_wins(M, N, K, cus, may_split)) ||
        (!aligned && few_tiles_count(M, N) < (1L << 31) && static_cast<long long>(M) * K >= 16 &&
         static_cast<long long>(N) * K >= 16)) {
      plan.cfg = 71;
      plan.splits = 0;
      return plan;
    }
    if (buf_ok) {
      switch (choose_tile(M, N, K, cus, false, may_split ? &auto_splits : nullptr)) {
        case Tile::kL8: plan.cfg = glb_ok ? 12 : 31; break;
        case Tile::kW128x2: plan.cfg = 41; break;
        case Tile::kM128x2: plan.cfg = 43; break;
        case Tile::kM128K2: plan.cfg = 53; break;
        case Tile::kS64x2: plan.cfg = 44; break;
        case Tile::kS64K2: plan.cfg = 51; break;
        case Tile::kR128K2: plan.cfg = 57; break;
        case Tile::kQ128K2: plan.cfg = 58; break;
        case Tile::kS64K4: plan.cfg = 59; break;
        case Tile::kW192K2: plan.cfg = 60; break;
        case Tile::kS64S4: plan.cfg = 33; break;
        case Tile::kM128S3: plan.cfg = 34; break;
        case Tile::kW128K2: case Tile::kW64x2: case Tile::kN32S3: case Tile::kN32K2:
          MXQ_CHECK(false, "a tile of gathered operands proposed for plain ones");
      }
    } else {
      if (tiles(256, 256) >= cus)
        plan.cfg = 1;
      else if (tiles(128, 128) >= cus)
        plan.cfg = 3;
      else
        plan.cfg = 4;
    }
    if (plan.splits == 0) plan.splits = auto_splits;
    // With the residual sum in the epilogue the balance moves (sweeps of every configuration
    // per layer inside the chained ResNet-50 body at batch 64): where the plain form takes
    // 256 x 128 tiles on 64-byte stages, 256 x 256 tiles on 128-byte stages are ahead once
    // they cover 0.56 of the CUs (12544 x 256 -> 1024: -1.9 us per layer) and 128 x 128
    // tiles otherwise (50176 x 128 -> 512: -1.2 us per layer).
    // The requantized sum is another third of arithmetic: 128 x 128 tiles throughout (12544 x 256
    // -> 1024 15.8 us against 16.8, 50176 x 128 -> 512 22.6 against 27.7).  (Where one round of 128 x 128 tiles
    // is proposed, on 128-byte stages, either form is level with 64-byte ones: 8192 x 320 -> 1024 10.5 and 11.0 us
    // against 10.7 and 11.1, 12544 x 320 -> 512 10.3 and 10.8 against 10.2 and 10.8.)
    if (sum && plan.cfg == 41) {
      if (!requant && K >= 256 && N > 128 && 16 * tiles(256, 256) >= 9 * cus)
        plan.cfg = 55;
      else
        plan.cfg = 43;
    }
    // The short-K streaming kernel, from 3 M outputs on (8192 x 64 -> 512 4.8 us against 5.4 on
    // tiles, 50176 x 128 -> 512 11.0 against 13.6, 50176 x 64 -> 1024 18.4 against 22.8; below,
    // the strips a work-group parks cost more than they save: 4096 x 128 -> 512 4.9 against 4.2,
    // 2048 x 128 -> 256 4.4 against 3.6).  128-column strips, three work-groups per CU, where an
    // output of 6 M gives every wave a few of them (50176 x 64 -> 256: 7.1 us against 7.2 on
    // 64-column strips, 50176 x 128 -> 512 11.0 against 11.9, 8192 x 64 -> 512 5.1 against 4.8).
    // With a sum the wide strips need the registers of two groups at K = 128 (50176 x 128 -> 512
    // 20.0 us, 21.4 on narrow ones, 21.2 on tiles), and at K <= 64 an output of 32 M (200704 x 64
    // -> 256 28.7 against 31.8 on narrow strips; 50176 rows 11.8 against 10.9).
    const int stream_rows = K == 256 ? 128 : 256;
    const bool stream_ok = aligned && fused8 && (K == 32 || K == 64 || K == 128 || K == 256) &&
                           N % 64 == 0 && (N <= stream_rows || N % stream_rows == 0);
    const long long outputs = static_cast<long long>(M) * N;
    if (stream_ok && K <= 128 && outputs >= 3LL << 20) {
      const bool wide = N % 128 == 0 && outputs >= (sum && K <= 64 ? 32LL << 20 : 6LL << 20);
      plan.cfg = wide ? 62 : 61;
      plan.splits = 1;
      if (force.stream_groups <= 0)
        plan.stream_groups = sum ? (wide && K > 64 ? 2 : 3) : (wide || K > 64 ? 3 : 4);
    }
  }
  if (plan.splits <= 0 && plan.cfg != 71) plan.splits = 1;
  return plan;
}

// Rows that are no multiple of 16 bytes: the few-tiles kernel reads them as they are, but a
// shape of many tiles is better copied into padded rows and given to the tiled kernels, where the
// caller brought room for the copies (K = 1237: 1024 x 1024 13.5 us against 11.2 with the copies,
// 256 x 2048 9.2 against 10.6).  Below 64 bytes a row there is little to read and the copies cost as much,
// so twice as many tiles are asked for (28717 x 18 -> 352, 9878 tiles, 38.9 us against 16.8; 136367 x 13
// -> 8, 4262 tiles, 19.7 against 15.5; 9245 x 58 -> 239, 2312 tiles, 16.7 against 12.6; 1813 x 19 -> 544,
// 969 tiles, 10.9 against 11.3).  However short they are: a copy sixteen times as large as rows of one
// byte is no larger than that of fifteen (60000 x 1 -> 16, 1875 tiles, 9.3 against 7.7, x 15 9.4 against 7.6; 60000 x 1
// -> 300 54 against 16.5, x 15 60 against 16.2).
int fc_padded_k(int M, int N, int K) {
  const int Kp = (K + 15) / 16 * 16;
  const bool wanted = Kp != K && few_tiles_count(M, N) > (K >= 64 ? 3L : 6L) * num_cus() &&
                      // (the copies read 16 bytes at once)
                      static_cast<long long>(M) * K >= 16 && static_cast<long long>(N) * K >= 16 &&
                      static_cast<long long>(M) * Kp < (1LL << 31) &&
                      static_cast<long long>(N) * Kp < (1LL << 31);
  return wanted ? Kp : 0;
}
size_t up256(long long x) { return static_cast<size_t>((x + 255) / 256 * 256); }
size_t fc_padded_bytes(int M, int N, int Kp) {
  return up256(static_cast<long long>(M) * Kp) + up256(static_cast<long long>(N) * Kp);
}

size_t fc_plan_workspace(const FcPlan& plan, int M, int N) {
  int bm, bn;
  if (plan.splits <= 1 || !fc_cfg_tile(plan.cfg, bm, bn)) return 0;
  const long tiles = static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  return splitk_workspace_bytes(tiles, plan.splits, bm, bn);
}

// ... with the workspace at hand: a split that the chooser proposed is dropped without room for it.
FcPlan plan_fc_within(int M, int N, int K, bool aligned, bool fused8, const GemmForce& force,
                      bool sum, bool requant, const Workspace& ws) {
  const FcPlan plan = plan_fc(M, N, K, aligned, fused8, force, sum, requant);
  if (force.splits != 0 || plan.splits <= 1 ||
      (ws.ptr != nullptr && aligned16(ws.ptr) && ws.bytes >= fc_plan_workspace(plan, M, N)))
    return plan;
  GemmForce unsplit = force;
  unsplit.splits = 1;
  return plan_fc(M, N, K, aligned, fused8, unsplit, sum, requant);
}

// Looks for a short form of the requantized sum over given ranges (SumPairs): the products of the
// rule's scales, each moved by up to three last places, the nearest first, until one gives the
// definition's result for every pair of int8 operands.  One work-group, sixteen quads
// of pairs per lane and candidate.  It runs when a plan is made, not per pass.
__global__ __launch_bounds__(1024) void sum_pairs_kernel(float layer_range,
                                                         float res_min, float res_max,
                                                         float min_calib, float max_calib,
                                                         SumPairs* out) {
  RequantRule r = sum_requant_rule(dev_maxabs(-layer_range, layer_range),
                                   dev_maxabs(res_min, res_max), min_calib, max_calib);
  const double level = static_cast<double>(r.in_scale) * static_cast<double>(r.qscale);
  const float ta = static_cast<float>(r.s0 * level), tb = static_cast<float>(r.s1 * level);
  auto moved = [](float v, int c) {  // c = 0, 1, 2, ...: 0, +1, -1, +2, ... last places
    return __int_as_float(__float_as_int(v) + ((c & 1) ? (c + 1) / 2 : -(c / 2)));
  };
  bool found = false;
  // no denormal, infinity or NaN among the candidates
  if (r.fast && ta > 1e-30f && tb > 1e-30f && ta < 1e30f && tb < 1e30f) {
    for (int c = 0; c < 49 && !found; ++c) {
      r.ta = moved(ta, c % 7);
      r.tb = moved(tb, c / 7);
      bool differs = false;
      for (int i = threadIdx.x; i < 64 * 256; i += 1024) {
        const int a0 = 4 * (i >> 8) - 127, b = (i & 255) - 128;  // a0 ... a0 + 3
        uint32_t x = 0;
        for (int k = 0; k < 4; ++k)  // -127 ... 127, the last quad one short
          x |= (static_cast<uint32_t>(a0 + k < 127 ? a0 + k : 127) & 0xffu) << (8 * k);
        const uint32_t y = (static_cast<uint32_t>(b) & 0xffu) * 0x01010101u;
        differs |= sum_pairs4(x, y, r) != sum_requant4_general<true>(x, y, r);
      }
      found = __syncthreads_or(differs) == 0;
    }
  }
  if (threadIdx.x == 0) {
    out->ta = r.ta;
    out->tb = r.tb;
    out->ok = found;
  }
}

// The scalars and the int32 bias of a layer whose ranges stay, the bits a launch computes itself.
__global__ __launch_bounds__(256) void prepare_layer_kernel(Epilogue e, int N, char* out) {
  const EpiScalars s = epi_scalars(e);
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n == 0) {
    *reinterpret_cast<EpiScalars*>(out) = s;
    *reinterpret_cast<LayerForms*>(out + kFormsAt) = LayerForms{0, 0.0f, 0.0f, 0.0f};
  }
  if (n < N) reinterpret_cast<int*>(out + kPreparedBias)[n] = epi_bias32(e, s, n);
}

// The layer's short forms into what prepare_layer_kernel wrote: a work-group each.
__global__ __launch_bounds__(1024) void prepare_forms_kernel(char* prepared) {
  __shared__ FormSearch search;
  const EpiScalars s = *reinterpret_cast<const EpiScalars*>(prepared);
  const bool relu = blockIdx.x == 0;
  const LayerForm f = find_form(s, relu, &search);
  if (threadIdx.x == 0 && f.has) {
    LayerForms* const out = reinterpret_cast<LayerForms*>(prepared + kFormsAt);
    if (relu) {
      out->t_relu = f.t;
      out->c_relu = f.c;
    } else {
      out->t_plain = f.t;
    }
    atomicOr(&out->has, relu ? 1 : 2);
  }
}

// an output without elements still owes its range scalars
__global__ void gemm_ranges_kernel(Epilogue e) { epilogue_ranges<kEpiSum>(e); }

void launch_fc(hipStream_t s, const int8_t* data, const int8_t* weight, int M, int N, int K,
               int ldo, const Epilogue& epi, const GemmForce& force, const Workspace& ws) {
  if (M == 0 || N == 0) {
    hipLaunchKernelGGL(gemm_ranges_kernel, dim3(1), dim3(1), 0, s, epi);
    MXQ_LAUNCH_CHECK();
    return;
  }
  FcArgs a;
  a.data = data;
  a.weight = weight;
  a.M = M;
  a.N = N;
  a.K = K;
  a.ldo = ldo;
  a.epi = epi;
  a.epi.stream8 = epi_stream_rows(M);
  a.sk.splits = 1;
  a.sk.kt_per_split = 1 << 30;
  a.sk.counters = nullptr;
  a.sk.partials = nullptr;
  const bool aligned = (K % 16 == 0) && aligned16(data) && aligned16(weight);
  // direct-to-LDS kernels: operands below 2 GiB; K a multiple of the 64-byte stage for
  // the global-load form, of 16 for the buffer-load form
  const bool buf_ok = aligned && K >= 16 && static_cast<long long>(M) * K < (1LL << 31) &&
                      static_cast<long long>(N) * K < (1LL << 31);
  const bool glb_ok = buf_ok && (K % 64 == 0);
  const bool fused8 = epi.out32 == nullptr && epi.outf == nullptr && epi.out8 != nullptr &&
                      ldo % 16 == 0 && aligned16(epi.out8) &&
                      (epi.res == nullptr || aligned16(epi.res));
  const bool sum = epi.res != nullptr;
  if (const int Kp = force.cfg == 0 && K % 16 != 0 ? fc_padded_k(M, N, K) : 0) {
    const size_t copies = fc_padded_bytes(M, N, Kp);
    if (ws.ptr != nullptr && aligned16(ws.ptr) && ws.bytes >= copies) {
      int8_t* d = static_cast<int8_t*>(ws.ptr);
      int8_t* w = d + up256(static_cast<long long>(M) * Kp);
      launch_pad_rows(s, data, M, d, weight, N, w, K, Kp);
      Workspace rest;
      rest.ptr = d + copies;
      rest.bytes = ws.bytes - copies;
      launch_fc(s, d, w, M, N, Kp, ldo, epi, force, rest);
      return;
    }
  }
  if ((force.cfg == 0 || force.cfg == 65) && (K == 256 || K == 512)) {  // its reductions
    ResidentArgs r = {};
    r.data = data;
    r.weight = weight;
    r.M = M;
    r.N = N;
    r.K = K;
    r.ldo = ldo;
    r.epi = a.epi;
    if (resident_wins(r, aligned && fused8)) {
      launch_resident(s, r);
      return;
    }
  }
  MXQ_CHECK(force.cfg != 65, "not a layer for the kernel with the weights in registers");
  const FcPlan plan =
      plan_fc_within(M, N, K, aligned, fused8, force, sum, epi.sum_requant != 0, ws);
  const int cfg = plan.cfg;
  if (cfg >= 11 && cfg <= 16) MXQ_CHECK(glb_ok, "shape does not qualify for the DMA kernels");
  if (cfg == 61 || cfg == 62) {
    const int stream_rows = K == 256 ? 128 : 256;  // weight rows one work-group parks in LDS
    const bool stream_ok = aligned && fused8 && (K == 32 || K == 64 || K == 128 || K == 256) &&
                           N % 64 == 0 && (N <= stream_rows || N % stream_rows == 0);
    MXQ_CHECK(stream_ok && (cfg == 61 || N % 128 == 0),
              "shape does not qualify for the short-K streaming kernel");
    MXQ_CHECK(plan.stream_groups >= 1 && plan.stream_groups <= 16, "stream_groups out of range");
  }
  if (cfg >= 21 && cfg < 61)
    MXQ_CHECK(buf_ok, "shape does not qualify for the buffer-load DMA kernels");
  if (cfg == 71) {
    FewTilesArgs f = {};
    f.data = data;
    f.weight = weight;
    f.M = M;
    f.N = N;
    f.K = K;
    f.ldo = ldo;
    f.epi = a.epi;
    launch_few_tiles_fc(s, f, buf_ok,
                        plan.splits != 0 ? plan.splits : few_tiles_waves(M, N, K, buf_ok));
    return;
  }
  if (cfg < 11) MXQ_CHECK(plan.splits <= 1, "the register-staged kernels have no split-K form");
  const FcLaunch how = {cfg, plan.splits, plan.stream_groups, aligned};
  switch (epi_mode(a.epi)) {
    case kEpiF32: fc_launch_f32(s, a, how, ws); break;
    case kEpiSum: fc_launch_sum(s, a, how, ws); break;
    case kEpiSumRq: fc_launch_sum_requant(s, a, how, ws); break;
    default: fc_launch_plain(s, a, how, ws);
  }
}

// Scratch bytes with which launch_fc takes its fastest route for this shape (0 when it
// would not split).  Assumes 16-byte aligned operands.  The residual-sum form plans its tile
// on its own (plan_fc's `sum`), so the figure is the larger of the two plans: a workspace
// sized by this query serves mxq_quantized_fc and mxq_quantized_fc_sum alike.
size_t fc_workspace_bytes(int M, int N, int K, bool fused8) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (const int Kp = K % 16 != 0 ? fc_padded_k(M, N, K) : 0)
    return fc_padded_bytes(M, N, Kp) + fc_workspace_bytes(M, N, Kp, fused8);
  const size_t plain =
      fc_plan_workspace(plan_fc(M, N, K, K % 16 == 0, fused8, GemmForce(), false), M, N);
  if (!fused8) return plain;
  const size_t sum =
      fc_plan_workspace(plan_fc(M, N, K, K % 16 == 0, true, GemmForce(), true), M, N);
  return plain > sum ? plain : sum;
}

}  // namespace mxq

using namespace mxq;

namespace {

// The residual sum fused behind the requantization (mxq_quantized_fc_sum).
struct SumArgs {
  const int8_t* res;
  const float* res_min;
  const float* res_max;
  float min_calib, max_calib;
  int relu;
  int requant;
  const SumPairs* pairs;
};

void fc_entry(void* stream, const int8_t* data, const int8_t* weight, const int8_t* bias, int M,
              int N, int K, const float* min_data, const float* max_data,
              const float* min_weight, const float* max_weight, const float* min_bias,
              const float* max_bias, int32_t* out32, float* omin, float* omax, int8_t* out8,
              float* out_f32, float* rmin, float* rmax, int relu, float min_calib,
              float max_calib, void* workspace, size_t workspace_bytes, const GemmForce& force,
              const SumArgs* sum = nullptr, const void* prepared = nullptr) {
  MXQ_CHECK(M >= 0 && N >= 0 && K >= 0, "negative dimension");
  if (prepared == nullptr) {
    MXQ_CHECK(min_data && max_data && min_weight && max_weight, "null input range pointer");
    MXQ_CHECK(omin && omax, "null output range pointer");
    MXQ_CHECK(bias == nullptr || (min_bias && max_bias), "bias given without its range");
    MXQ_CHECK((out8 == nullptr && out_f32 == nullptr) || (rmin && rmax),
              "fused requantize needs rmin/rmax");
  }
  MXQ_CHECK(M == 0 || N == 0 || out32 != nullptr || out8 != nullptr || out_f32 != nullptr,
            "no output buffer");
  MXQ_CHECK(M == 0 || N == 0 || K == 0 || (data != nullptr && weight != nullptr),
            "null operand pointer");
  Epilogue e;
  e.bias = bias;
  e.min_data = min_data;
  e.max_data = max_data;
  e.min_weight = min_weight;
  e.max_weight = max_weight;
  e.min_bias = min_bias;
  e.max_bias = max_bias;
  e.out32 = out32;
  e.out8 = out8;
  e.outf = out_f32;
  e.res = nullptr;
  e.res_min = e.res_max = nullptr;
  e.sum_min_calib = e.sum_max_calib = 0.f;
  e.sum_relu = 0;
  e.sum_requant = 0;
  e.sum_pairs = nullptr;
  e.with_sum = 0;
  if (sum != nullptr) {
    MXQ_CHECK((M == 0 || N == 0 || out8 != nullptr) && out32 == nullptr && out_f32 == nullptr,
              "the fused sum writes the int8 output only");
    MXQ_CHECK(sum->res_min && sum->res_max, "null residual range pointer");
    MXQ_CHECK(M == 0 || N == 0 || sum->res != nullptr, "null residual operand");
    if (M != 0 && N != 0) {  // without elements only the ranges are written
      e.res = sum->res;
      e.res_min = sum->res_min;
      e.res_max = sum->res_max;
    }
    e.sum_min_calib = sum->min_calib;
    e.sum_max_calib = sum->max_calib;
    e.sum_relu = sum->relu;
    e.sum_requant = sum->requant;
    e.sum_pairs = sum->pairs;
    e.with_sum = 1;
  }
  e.prepared = static_cast<const char*>(prepared);
  e.omin = omin;
  e.omax = omax;
  e.rmin = rmin;
  e.rmax = rmax;
  e.relu = relu;
  float a = fabsf(min_calib), b = fabsf(max_calib);
  e.real_range = (a < b) ? b : a;
  e.plane = 0;
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  launch_fc(static_cast<hipStream_t>(stream), data, weight, M, N, K, N, e, force, ws);
}

}  // namespace

extern "C" {

size_t mxq_quantized_fc_workspace(int M, int N, int K, int fused_int8_only) {
  try {
    return fc_workspace_bytes(M, N, K, fused_int8_only != 0 && N % 16 == 0);
  } catch (...) {
    return 0;
  }
}

int mxq_quantized_fc(void* stream, const int8_t* data, const int8_t* weight, const int8_t* bias,
                     int M, int N, int K, const float* min_data, const float* max_data,
                     const float* min_weight, const float* max_weight, const float* min_bias,
                     const float* max_bias, int32_t* out32, float* omin, float* omax,
                     int8_t* out8, float* rmin, float* rmax, int relu, float min_calib,
                     float max_calib, void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, out32, omin, omax, out8, nullptr, rmin, rmax, relu, min_calib,
           max_calib, workspace, workspace_bytes, GemmForce());
  MXQ_API_END();
}

#ifdef MXQ_TEST_HOOKS
// Test-only twin of mxq_quantized_fc (declared in tests/mxq_test_hooks.h, not in the
// operator header): the tile configuration, the split-K factor and the streaming kernel's
// work-groups per CU come as arguments (0 = let the launcher choose), so tests can drive
// every kernel variant on any shape without process-wide state.
int mxq_test_quantized_fc(void* stream, const int8_t* data, const int8_t* weight,
                          const int8_t* bias, int M, int N, int K, const float* min_data,
                          const float* max_data, const float* min_weight,
                          const float* max_weight, const float* min_bias, const float* max_bias,
                          int32_t* out32, float* omin, float* omax, int8_t* out8, float* rmin,
                          float* rmax, int relu, float min_calib, float max_calib,
                          void* workspace, size_t workspace_bytes, int cfg, int splits,
                          int stream_groups) {
  MXQ_API_BEGIN();
  GemmForce force;
  force.cfg = cfg;
  force.splits = splits;
  force.stream_groups = stream_groups;
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, out32, omin, omax, out8, nullptr, rmin, rmax, relu, min_calib,
           max_calib, workspace, workspace_bytes, force);
  MXQ_API_END();
}

// tests/mxq_test_hooks.h
int mxq_test_fc_plan(int M, int N, int K, int fused_int8, int sum, int requant, void* workspace,
                     size_t workspace_bytes, int* cfg, int* splits) {
  MXQ_API_BEGIN();
  MXQ_CHECK(M > 0 && N > 0 && K > 0 && cfg != nullptr && splits != nullptr, "bad arguments");
  Workspace ws;
  ws.ptr = workspace;
  ws.bytes = workspace_bytes;
  const FcPlan plan = plan_fc_within(M, N, K, K % 16 == 0, fused_int8 != 0, GemmForce(), sum != 0,
                                     requant != 0, ws);
  *cfg = plan.cfg;
  *splits = plan.splits;
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

int mxq_quantized_fc_f32(void* stream, const int8_t* data, const int8_t* weight,
                         const int8_t* bias, int M, int N, int K, const float* min_data,
                         const float* max_data, const float* min_weight, const float* max_weight,
                         const float* min_bias, const float* max_bias, float* out_f32,
                         float* omin, float* omax, float* rmin, float* rmax, int relu,
                         float min_calib, float max_calib, void* workspace,
                         size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(M == 0 || N == 0 || out_f32 != nullptr, "no output buffer");
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, nullptr, out_f32, rmin, rmax, relu,
           min_calib, max_calib, workspace, workspace_bytes, GemmForce());
  MXQ_API_END();
}

int mxq_quantized_fc_sum(void* stream, const int8_t* data, const int8_t* weight,
                         const int8_t* bias, int M, int N, int K, const float* min_data,
                         const float* max_data, const float* min_weight, const float* max_weight,
                         const float* min_bias, const float* max_bias, const int8_t* residual,
                         const float* min_residual, const float* max_residual, int8_t* out8,
                         float* omin, float* omax, float* rmin, float* rmax, float min_calib,
                         float max_calib, float sum_min_calib, float sum_max_calib, int sum_relu,
                         void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  const SumArgs sum = {residual, min_residual, max_residual, sum_min_calib, sum_max_calib,
                       sum_relu, 0, nullptr};
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, out8, nullptr, rmin, rmax, 0, min_calib,
           max_calib, workspace, workspace_bytes, GemmForce(), &sum);
  MXQ_API_END();
}

int mxq_quantized_fc_sum_requant(void* stream, const int8_t* data, const int8_t* weight,
                                 const int8_t* bias, int M, int N, int K, const float* min_data,
                                 const float* max_data, const float* min_weight,
                                 const float* max_weight, const float* min_bias,
                                 const float* max_bias, const int8_t* residual,
                                 const float* min_residual, const float* max_residual,
                                 int8_t* out8, float* omin, float* omax, float* rmin, float* rmax,
                                 float min_calib, float max_calib, float sum_min_calib,
                                 float sum_max_calib, int sum_relu, const void* pairs,
                                 void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK((reinterpret_cast<uintptr_t>(pairs) & 3u) == 0, "unaligned pairs");
  const SumArgs sum = {residual, min_residual, max_residual, sum_min_calib, sum_max_calib,
                       sum_relu, 1, static_cast<const SumPairs*>(pairs)};
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, out8, nullptr, rmin, rmax, 0, min_calib,
           max_calib, workspace, workspace_bytes, GemmForce(), &sum);
  MXQ_API_END();
}

int mxq_prepare_layer(void* stream, const int8_t* bias, int N, const float* min_data,
                      const float* max_data, const float* min_weight, const float* max_weight,
                      const float* min_bias, const float* max_bias, float min_calib,
                      float max_calib, void* prepared) {
  MXQ_API_BEGIN();
  MXQ_CHECK(N >= 0, "negative dimension");
  MXQ_CHECK(min_data && max_data && min_weight && max_weight, "null input range pointer");
  MXQ_CHECK(bias == nullptr || (min_bias && max_bias), "bias given without its range");
  MXQ_CHECK(prepared != nullptr && aligned16(prepared), "null or unaligned pointer");
  Epilogue e = {};
  e.bias = bias;
  e.min_data = min_data;
  e.max_data = max_data;
  e.min_weight = min_weight;
  e.max_weight = max_weight;
  e.min_bias = min_bias;
  e.max_bias = max_bias;
  const float a = fabsf(min_calib), b = fabsf(max_calib);
  e.real_range = (a < b) ? b : a;
  hipLaunchKernelGGL(prepare_layer_kernel, dim3(static_cast<unsigned>(N / 256 + 1)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), e, N, static_cast<char*>(prepared));
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_prepare_forms(void* stream, void* prepared) {
  MXQ_API_BEGIN();
  MXQ_CHECK(prepared != nullptr && aligned16(prepared), "null or unaligned pointer");
  hipLaunchKernelGGL(prepare_forms_kernel, dim3(2), dim3(1024), 0, static_cast<hipStream_t>(stream),
                     static_cast<char*>(prepared));
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_quantized_fc_prepared(void* stream, const int8_t* data, const int8_t* weight,
                              const void* prepared, int M, int N, int K, int8_t* out8,
                              float* out_f32, int relu, float min_calib, float max_calib,
                              void* workspace, size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(prepared != nullptr && aligned16(prepared), "null or unaligned pointer");
  MXQ_CHECK((out8 == nullptr) != (out_f32 == nullptr), "one output buffer");
  fc_entry(stream, data, weight, nullptr, M, N, K, nullptr, nullptr, nullptr, nullptr, nullptr,
           nullptr, nullptr, nullptr, nullptr, out8, out_f32, nullptr, nullptr, relu, min_calib,
           max_calib, workspace, workspace_bytes, GemmForce(), nullptr, prepared);
  MXQ_API_END();
}

int mxq_quantized_fc_sum_prepared(void* stream, const int8_t* data, const int8_t* weight,
                                  const void* prepared, int M, int N, int K,
                                  const int8_t* residual, const float* min_residual,
                                  const float* max_residual, int8_t* out8, float min_calib,
                                  float max_calib, float sum_min_calib, float sum_max_calib,
                                  int sum_relu, int requant, const void* pairs, void* workspace,
                                  size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(prepared != nullptr && aligned16(prepared), "null or unaligned pointer");
  MXQ_CHECK((reinterpret_cast<uintptr_t>(pairs) & 3u) == 0, "unaligned pairs");
  const SumArgs sum = {residual, min_residual, max_residual, sum_min_calib, sum_max_calib,
                       sum_relu, requant, requant ? static_cast<const SumPairs*>(pairs) : nullptr};
  fc_entry(stream, data, weight, nullptr, M, N, K, nullptr, nullptr, nullptr, nullptr, nullptr,
           nullptr, nullptr, nullptr, nullptr, out8, nullptr, nullptr, nullptr, 0, min_calib,
           max_calib, workspace, workspace_bytes, GemmForce(), &sum, prepared);
  MXQ_API_END();
}

int mxq_sum_requant_pairs(void* stream, float min_calib, float max_calib,
                          float min_residual, float max_residual, float sum_min_calib,
                          float sum_max_calib, void* pairs) {
  MXQ_API_BEGIN();
  MXQ_CHECK(pairs != nullptr, "null pointer");
  MXQ_CHECK((reinterpret_cast<uintptr_t>(pairs) & 3u) == 0, "unaligned pairs");
  const float a = fabsf(min_calib), b = fabsf(max_calib);
  hipLaunchKernelGGL(sum_pairs_kernel, dim3(1), dim3(1024), 0, static_cast<hipStream_t>(stream),
                     (a < b) ? b : a, min_residual, max_residual, sum_min_calib, sum_max_calib,
                     static_cast<SumPairs*>(pairs));
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

#ifdef MXQ_TEST_HOOKS
// Test-only twins of the two residual-sum entry points with the kernel variant pinned
// (tests/mxq_test_hooks.h).
int mxq_test_quantized_fc_sum(void* stream, const int8_t* data, const int8_t* weight,
                              const int8_t* bias, int M, int N, int K, const float* min_data,
                              const float* max_data, const float* min_weight,
                              const float* max_weight, const float* min_bias,
                              const float* max_bias, const int8_t* residual,
                              const float* min_residual, const float* max_residual,
                              int8_t* out8, float* omin, float* omax, float* rmin, float* rmax,
                              float min_calib, float max_calib, float sum_min_calib,
                              float sum_max_calib, int sum_relu, void* workspace,
                              size_t workspace_bytes, int cfg, int splits, int stream_groups) {
  MXQ_API_BEGIN();
  const SumArgs sum = {residual, min_residual, max_residual, sum_min_calib, sum_max_calib,
                       sum_relu, 0, nullptr};
  GemmForce force;
  force.cfg = cfg;
  force.splits = splits;
  force.stream_groups = stream_groups;
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, out8, nullptr, rmin, rmax, 0, min_calib,
           max_calib, workspace, workspace_bytes, force, &sum);
  MXQ_API_END();
}

int mxq_test_quantized_fc_sum_requant(void* stream, const int8_t* data, const int8_t* weight,
                              const int8_t* bias, int M, int N, int K, const float* min_data,
                              const float* max_data, const float* min_weight,
                              const float* max_weight, const float* min_bias,
                              const float* max_bias, const int8_t* residual,
                              const float* min_residual, const float* max_residual,
                              int8_t* out8, float* omin, float* omax, float* rmin, float* rmax,
                              float min_calib, float max_calib, float sum_min_calib,
                              float sum_max_calib, int sum_relu, const void* pairs,
                              void* workspace, size_t workspace_bytes, int cfg, int splits, int stream_groups) {
  MXQ_API_BEGIN();
  const SumArgs sum = {residual, min_residual, max_residual, sum_min_calib, sum_max_calib,
                       sum_relu, 1, static_cast<const SumPairs*>(pairs)};
  GemmForce force;
  force.cfg = cfg;
  force.splits = splits;
  force.stream_groups = stream_groups;
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, out8, nullptr, rmin, rmax, 0, min_calib,
           max_calib, workspace, workspace_bytes, force, &sum);
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

#ifdef MXQ_TEST_HOOKS
// Test-only twin of mxq_quantized_fc_f32 with the tile configuration and the split-K factor
// pinned (tests/mxq_test_hooks.h).
int mxq_test_quantized_fc_f32(void* stream, const int8_t* data, const int8_t* weight,
                              const int8_t* bias, int M, int N, int K, const float* min_data,
                              const float* max_data, const float* min_weight,
                              const float* max_weight, const float* min_bias,
                              const float* max_bias, float* out_f32, float* omin, float* omax,
                              float* rmin, float* rmax, int relu, float min_calib,
                              float max_calib, void* workspace, size_t workspace_bytes, int cfg,
                              int splits) {
  MXQ_API_BEGIN();
  MXQ_CHECK(M == 0 || N == 0 || out_f32 != nullptr, "no output buffer");
  GemmForce force;
  force.cfg = cfg;
  force.splits = splits;
  force.stream_groups = 0;
  fc_entry(stream, data, weight, bias, M, N, K, min_data, max_data, min_weight, max_weight,
           min_bias, max_bias, nullptr, omin, omax, nullptr, out_f32, rmin, rmax, relu,
           min_calib, max_calib, workspace, workspace_bytes, force);
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

}  // extern "C"
