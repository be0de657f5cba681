// 1 x 1 convolutions (of any stride) and fully-connected layers with an int8 output, a reduction
// of 256 or 512 bytes and many rows.
//
// A tile of the other kernels is at most 8 K steps here: it fetches its weights again, waits for a
// first stage, and ends in an epilogue that the matrix units stand still for.  A work-group of this
// one stays on its columns: their weights are loaded once, into registers, and row tiles stream
// past them through LDS, three or four on their way (vmcnt counts them and the stores, one order),
// one barrier each; a tile's bytes leave one tile later, as whole rows of the group's columns.
// Two groups of four waves share a CU, so that one's epilogue meets the other's products; four
// waves per SIMD on half as many columns each read the rows from LDS twice as often and are level.
//
// What is left to bound it: the epilogue's 6.7 VALU instructions per output and the products do not
// overlap (50176 rows of 256 -> 512: 15.0 us, of which 5.3 are HBM).  us, rows of K -> N, on tiles
// / here, one launch in a chain over inputs of more than the caches hold:
//   50176 x 256 -> 512    19.0 / 15.0     200704 x 256 -> 64    19.8 / 14.9
//   200704 x 256 -> 512   66.5 / 49.0     50176 x 256 -> 128     8.6 /  7.8
//   12544 x 256 -> 1024   10.1 / 10.0     50176 x 512 -> 128    12.2 / 10.8
//   50176 x 256 -> 1024   34.1 / 25.1     50176 x 512 -> 256    17.1 / 16.0
//   12544 x 512 -> 1024   14.5 / 14.4     50176 x 512 -> 512    30.8 / 24.1
//   50176 x 512 -> 1024   52.5 / 38.9
// With 1.5 tiles a group the weights' way in costs what is saved (12544 x 512 -> 512 9.2 / 10.4,
// 12544 x 512 -> 256 7.4 / 8.2; 256 bytes: level), hence the rule.  A reduction of 128 bytes stays
// with fc_stream_kernel (50176 x 128 -> 512 12.0, here 12.1).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_forms.h"
#include "mxq_resident.h"

namespace mxq {
namespace {

constexpr int kNonTemporal = 2;  // the buffer instructions' nt bit

// n / d for n * d < 2^30, magic = 2^31 / d + 1
__device__ __forceinline__ int quotient(int n, uint32_t magic) {
  return static_cast<int>(__umulhi(2u * static_cast<uint32_t>(n) + 1u, magic));
}
uint32_t magic_of(int d) {
  return static_cast<uint32_t>((1ULL << 31) / static_cast<unsigned>(d) + 1);
}

struct Args {
  ResidentArgs r;
  uint32_t magic_area, magic_ow;
  int step_images, step_rest;  // the rows between two tiles of a work-group, by images
};

constexpr int kRing = 8192;  // bytes in LDS through which a wave's weights come

// 4 waves, WN of them side by side, each on 32 rows and NI times 32 columns of a tile; NS tiles of
// operand rows in LDS, two work-groups per CU.
template <int KS, int WN, int NI, int NS, bool GATHER, bool FORMS = false>
__device__ __forceinline__ void resident(const Args& args, const ResidentArgs& p, int group) {
  constexpr int NW = 4, THREADS = 64 * NW, WM = NW / WN, TM = 32 * WM, TN = 32 * NI, NC = WN * TN;
  constexpr int K = 32 * KS, CH = 2 * KS;
  constexpr int D = TM * CH / THREADS;           // DMA instructions of a wave and tile
  constexpr int S = TM * NC / 16 / THREADS;      // stores of a lane and tile
  constexpr int LD = NC + 16, PIECES = NC / 16;
  static_assert(D >= 1 && S >= 1, "tile too small");
  static_assert(2 * TM * LD + NC * 4 <= NW * kRing, "the rings' place is too small");
  static_assert(NS * TM * CH * 16 + NW * kRing <= 80 * 1024, "LDS of two work-groups");
  __shared__ __attribute__((aligned(16))) v4i rows[NS * TM * CH];
  // first the weights' rings, then two output tiles and the bias
  __shared__ __attribute__((aligned(16))) char shared[NW * kRing];
  char* const out = shared;
  int* const bias = reinterpret_cast<int*>(shared + 2 * TM * LD);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, lrow = lane & 31, lgrp = lane >> 5;
  const int n0 = group * NC;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(rows));
  auto swizzle = [](int r) { return CH == 4 ? (r >> 2) & 3 : r & 15; };

  // the rows' way into LDS: lane's slot (row, chunk) holds chunk ^ swizzle(row) of that row
  int m_next = blockIdx.x * TM;            // first row of the tile that is fetched next
  const int m_step = gridDim.x * TM;
  int image = 0, rest = 0;                 // m_next by images
  if (GATHER) {
    image = m_next / p.area;
    rest = m_next - image * p.area;
  }
  int slot_row[D], slot_chunk[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int slot = (d * NW + wave) * 64 + lane;
    slot_row[d] = slot / CH;
    slot_chunk[d] = ((slot % CH) ^ swizzle(slot / CH)) * 16;
  }
  auto fetch = [&](int stage) {
    const int left = p.M - m_next;
    const int8_t* base = p.data;
    long long bytes = 0;
    if (left > 0) {
      if (GATHER) {
        base += image * p.image;
        bytes = (p.images - image) * p.image;
      } else {
        base += static_cast<long long>(m_next) * K;
        bytes = static_cast<long long>(left) * K;
      }
    }
    const v4i rsrc =
        make_rsrc(base, bytes < 0x7fffffff ? static_cast<uint32_t>(bytes) : 0x7fffffffu);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      uint32_t at;
      if (GATHER) {
        const int x = rest + slot_row[d], img = quotient(x, args.magic_area);
        const int y = x - img * p.area, oh = quotient(y, args.magic_ow);
        at = static_cast<uint32_t>(img * static_cast<int>(p.image) + oh * p.down +
                                   (y - oh * p.OW) * p.right + slot_chunk[d]);
        at = slot_row[d] < left ? at : kOutOfRange;
      } else {
        at = static_cast<uint32_t>(slot_row[d] * K + slot_chunk[d]);
      }
      const uint32_t to = lds0 + (stage * TM * CH + (d * NW + wave) * 64) * 16;
      dma_buffer(__builtin_amdgcn_readfirstlane(to), at, rsrc);
    }
    m_next += m_step;
    if (GATHER) {
      image += args.step_images;
      rest += args.step_rest;
      if (rest >= p.area) {
        rest -= p.area;
        ++image;
      }
    }
  };
  // What leaves of a tile: 16-byte pieces, whole rows of the work-group's columns.  A tile without
  // rows stores nothing but counts the same.
  auto store = [&](int m0, const char* from, auto stream) {
    const int left = p.M - m0;
    const int height = m0 < 0 ? 0 : left < TM ? (left > 0 ? left : 0) : TM;
    const int8_t* const base =
        height > 0 ? p.epi.out8 + static_cast<size_t>(m0) * p.ldo + n0 : p.epi.out8;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(base), 0, height > 0 ? (height - 1) * p.ldo + p.N - n0 : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int piece = i * THREADS + tid, row = piece / PIECES, c = piece % PIECES;
      const v4i v = *reinterpret_cast<const v4i*>(from + row * LD + c * 16);
      const uint32_t at =
          n0 + c * 16 < p.N ? static_cast<uint32_t>(row * p.ldo + c * 16) : kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, at, 0,
                                             decltype(stream)::value ? kNonTemporal : kDeviceScope);
    }
  };

  // the first tiles, then everything else that is loaded once
#pragma unroll
  for (int j = 0; j < NS - 1; ++j) fetch(j);
  // The wave's weights, as the matrix instructions take them: column n's K bytes over a lane pair.
  // Loaded like that an instruction would touch 32 lines for 32 bytes of each (4.6 us for 256
  // columns of 256 bytes); whole lines go through LDS instead, 128 bytes of 32 columns at a time.
  v4i weight[NI][KS];
  {
    // pieces of up to 128 bytes of 32 columns, a few instructions each
    constexpr int STEPS = KS < 4 ? KS : 4, RC = 2 * STEPS, ASKS = RC / 2, PARTS = KS / STEPS;
    constexpr int UNITS = NI * PARTS;
    static_assert(UNITS >= 2, "both places of the ring");
    const v4i rsrc = make_rsrc(p.weight, static_cast<uint32_t>(p.N) * K);
    const int first = n0 + wn * TN;
    const uint32_t ring = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(shared)) + wave * kRing;
    const v4i* const held = reinterpret_cast<const v4i*>(shared + wave * kRing);
    auto mixed = [](int r) { return RC == 4 ? (r >> 2) & 3 : (r ^ (r >> 2)) & 7; };
    auto ask = [&](int u) {
      const int ni = u / PARTS, part = u % PARTS;
#pragma unroll
      for (int i = 0; i < ASKS; ++i) {
        const int r = i * (64 / RC) + lane / RC, c = (lane % RC) ^ mixed(r);
        dma_buffer(__builtin_amdgcn_readfirstlane(ring + (u % 2) * 4096 + i * 1024),
                   static_cast<uint32_t>((first + ni * 32 + r) * K + part * 128 + c * 16), rsrc);
      }
    };
    ask(0);
    ask(1);
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      if (u + 1 < UNITS)
        wait_vmcnt<ASKS>();
      else
        wait_vmcnt<0>();
#pragma unroll
      for (int k = 0; k < STEPS; ++k)
        weight[u / PARTS][u % PARTS * STEPS + k] =
            held[(u % 2) * 256 + lrow * RC + ((k * 2 + lgrp) ^ mixed(lrow))];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (u + 2 < UNITS) ask(u + 2);
    }
  }
  const EpiScalars s = epi_scalars(p.epi);
  __syncthreads();  // the rings' place is the bias's from here on
  for (int i = tid; i < NC; i += THREADS) bias[i] = n0 + i < p.N ? epi_bias32(p.epi, s, n0 + i) : 0;
  __syncthreads();
  v16i held_bias[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      const v4i b = *reinterpret_cast<const v4i*>(bias + wn * TN + ni * 32 + 8 * vq + 4 * lgrp);
#pragma unroll
      for (int i = 0; i < 4; ++i) held_bias[ni][4 * vq + i] = b[i];
    }
    asm volatile("" : "+v"(held_bias[ni]));
  }
  LayerForms forms = {};
  if constexpr (FORMS) forms = *reinterpret_cast<const LayerForms*>(p.epi.prepared + kFormsAt);
  auto run = [&](auto stream, auto relu, auto short_form) {
    int stage = 0, ahead = NS - 1, before = -1, parity = 0;
    for (int m0 = blockIdx.x * TM; m0 < p.M; m0 += m_step) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S + (NS - 2) * (D + S))
                   : "memory");
      fetch(ahead);
      store(before, out + (parity ^ 1) * TM * LD, stream);
      v16i acc[NI];
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) acc[ni] = held_bias[ni];
      const v4i* const a = rows + stage * TM * CH + (wm * 32 + lrow) * CH;
      const int sw = swizzle(wm * 32 + lrow);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const v4i fa = a[(ks * 2 + lgrp) ^ sw];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          acc[ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(weight[ni][ks], fa, acc[ni], 0, 0, 0);
      }
      char* const to = out + parity * TM * LD + (wm * 32 + lrow) * LD + wn * TN + 4 * lgrp;
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
        {
          const int a0 = acc[ni][4 * vq], a1 = acc[ni][4 * vq + 1], a2 = acc[ni][4 * vq + 2],
                    a3 = acc[ni][4 * vq + 3];
          uint32_t w;
          if constexpr (!decltype(short_form)::value)
            w = epi_requant_pack<decltype(relu)::value>(a0, a1, a2, a3, s);
          else if constexpr (decltype(relu)::value)
            w = short_relu4(a0, a1, a2, a3, forms.t_relu, forms.c_relu);
          else
            w = short_plain4(a0, a1, a2, a3, forms.t_plain);
          *reinterpret_cast<uint32_t*>(to + ni * 32 + 8 * vq) = w;
        }
      before = m0;
      parity ^= 1;
      stage = stage + 1 == NS ? 0 : stage + 1;
      ahead = ahead + 1 == NS ? 0 : ahead + 1;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    store(before, out + (parity ^ 1) * TM * LD, stream);
  };
  typedef std::true_type Yes;
  typedef std::false_type No;
  auto run_form = [&](auto stream) {
    if constexpr (FORMS) {
      if (p.epi.relu && (forms.has & 1)) {
        run(stream, Yes(), Yes());
        return;
      }
      if (!p.epi.relu && (forms.has & 2)) {
        run(stream, No(), Yes());
        return;
      }
    }
    if (p.epi.relu)
      run(stream, Yes(), No());
    else
      run(stream, No(), No());
  };
  if (p.epi.stream8)
    run_form(Yes());
  else
    run_form(No());
  if (blockIdx.x == 0 && group == 0 && tid == 0) epilogue_ranges<kEpiPlain>(p.epi);
}

template <int KS, int WN, int NI, int NS, bool GATHER>
__global__ __launch_bounds__(256, 2) void resident_kernel(Args args) {
  resident<KS, WN, NI, NS, GATHER>(args, args.r, blockIdx.y);
}

// Two layers over the same rows: the stage starts of a network, whose first layer and projection read
// the same tensor.  Their scales stay, so the requantize takes its short form where one was found
// (mxq_forms.h): 4 instead of 7.75 vector instructions an output without a relu, 3.25 instead of
// 6.7 with it.  Batch 64, us, two launches / one launch / with the short forms:
//   200704 x 64 -> 64 and 256   27.0 / - / 20.0      50176 x 256 -> 128 and 512  26.2 / 24.0 / 19.3
//   12544 x 512 -> 256 and 1024 26.6 / 20.4 / 18.3
struct PairArgs {
  Args a;
  ResidentArgs b;
  int first;  // column groups of the first
};
template <int KS, int WN, int NS, bool GATHER>
__global__ __launch_bounds__(256, 2) void resident_pair_kernel(PairArgs args) {
  const bool second = static_cast<int>(blockIdx.y) >= args.first;
  ResidentArgs r = args.a.r;
  if (second) r = args.b;
  resident<KS, WN, 2, NS, GATHER, true>(args.a, r,
                                        static_cast<int>(blockIdx.y) - (second ? args.first : 0));
}

// Work-groups along the rows, and how a tile's images follow the one before.
int row_groups(Args& a, int tile, int column_groups) {
  const ResidentArgs& r = a.r;
  const int tiles = (r.M + tile - 1) / tile;
  int gx = 2 * num_cus() / column_groups;
  if (gx > 8) gx = gx / 8 * 8;  // column groups of the same rows on the same XCD
  if (gx < 1) gx = 1;
  if (gx > tiles) gx = tiles;
  if (r.area != 0) {
    const long long step = static_cast<long long>(gx) * tile;
    a.magic_area = magic_of(r.area);
    a.magic_ow = magic_of(r.OW);
    a.step_images = static_cast<int>(step / r.area);
    a.step_rest = static_cast<int>(step % r.area);
  }
  return gx;
}

template <int KS, int WN, int NI, int NS>
void launch(hipStream_t s, Args& a) {
  constexpr int NC = 32 * WN * NI;
  const int ny = (a.r.N + NC - 1) / NC, gx = row_groups(a, 128 / WN, ny);
  if (a.r.area != 0)
    hipLaunchKernelGGL((resident_kernel<KS, WN, NI, NS, true>), dim3(gx, ny), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((resident_kernel<KS, WN, NI, NS, false>), dim3(gx, ny), dim3(256), 0, s, a);
  MXQ_LAUNCH_CHECK();
}

// Columns of a work-group and rows of a tile of a pair.
int pair_columns(int K) { return K == 64 ? 128 : 256; }
int pair_rows(int K) { return K == 64 ? 64 : 32; }

template <int KS, int WN, int NS>
void launch_pair(hipStream_t s, PairArgs& p) {
  constexpr int NC = 64 * WN;
  const int first = (p.a.r.N + NC - 1) / NC, ny = first + (p.b.N + NC - 1) / NC;
  const int gx = row_groups(p.a, 128 / WN, ny);
  p.first = first;
  if (p.a.r.area != 0)
    hipLaunchKernelGGL((resident_pair_kernel<KS, WN, NS, true>), dim3(gx, ny), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((resident_pair_kernel<KS, WN, NS, false>), dim3(gx, ny), dim3(256), 0, s, p);
  MXQ_LAUNCH_CHECK();
}

bool takes(const ResidentArgs& a, bool aligned) {
  if (!aligned || a.epi.out8 == nullptr || a.epi.out32 != nullptr || a.epi.outf != nullptr ||
      a.epi.with_sum)
    return false;
  if (a.N % 16 != 0) return false;
  if (static_cast<long long>(a.N) * a.K >= (1LL << 31) || a.ldo >= (1 << 24)) return false;
  if (a.area != 0) {
    // what quotient() and the offsets inside a tile hold
    const long long span = (128 / a.area + 2) * a.image;
    if (a.area >= 30000 || a.OW >= 30000 || span >= (1LL << 31)) return false;
  }
  return true;
}

}  // namespace

bool resident_wins(const ResidentArgs& a, bool aligned) {
  if (!takes(a, aligned) || (a.K != 256 && a.K != 512)) return false;
  const int wide = a.K == 256 && a.N <= 64 ? 64 : a.N <= 128 ? 128 : 256;  // columns of a group
  const int high = wide == 64 ? 64 : 32;                                   // rows of a tile
  const long long groups = (a.N + wide - 1) / wide, tiles = (a.M + high - 1LL) / high * groups;
  if (4 * a.N < 3 * groups * wide) return false;
  return tiles >= (a.K == 256 ? 3 : 6) * num_cus();
}

bool resident_pair_wins(const ResidentArgs& a, const ResidentArgs& b, bool aligned) {
  if (!takes(a, aligned) || !takes(b, aligned)) return false;
  if (a.K != 64 && a.K != 256 && a.K != 512) return false;
  const int wide = pair_columns(a.K), high = pair_rows(a.K);
  const long long groups = (a.N + wide - 1) / wide + (b.N + wide - 1) / wide;
  if (3 * (a.N + b.N) < 2 * groups * wide) return false;
  return (a.M + high - 1LL) / high * groups >= (a.K == 512 ? 6 : 3) * num_cus();
}

void launch_resident_pair(hipStream_t s, const ResidentArgs& a, const ResidentArgs& b) {
  PairArgs p = {};
  p.a.r = a;
  p.b = b;
  if (a.K == 64) launch_pair<2, 2, 3>(s, p);
  else if (a.K == 256) launch_pair<8, 4, 4>(s, p);
  else launch_pair<16, 4, 3>(s, p);
}

void launch_resident(hipStream_t s, const ResidentArgs& r) {
  Args a = {};
  a.r = r;
  if (r.K == 256) {
    if (r.N <= 64) launch<8, 2, 1, 3>(s, a);
    else if (r.N <= 128) launch<8, 4, 1, 4>(s, a);
    else launch<8, 4, 2, 4>(s, a);
  } else {
    if (r.N <= 128) launch<16, 4, 1, 3>(s, a);
    else launch<16, 4, 2, 3>(s, a);
  }
}

}  // namespace mxq
