// The tail of a residual block as one launch: 3 x 3 convolution, 1 x 1 convolution, the sum with
// the shortcut, and the next block's first 1 x 1 convolution, each with its requantize and relu.
//
// Layer by layer every one of these is a launch of 10 to 30 us around 2 to 6 us of matrix work:
// its operands come through memory, its K loop waits for a stage at every barrier, its epilogue
// leaves the matrix cores idle.  The 1 x 1 layers need nothing but the pixels of the layer in
// front of them, so a work-group that owns whole pixels (all channels of TM consecutive ones)
// keeps them in LDS from the 3 x 3 layer's input to the last layer's output:
//
//   patch   the input rows its pixels touch, halo included          [rows][W + 2][C]
//           then the 3 x 3 layer's int8 result                      [TM][Cm]
//           then the next block's first layer                       [TM][Ca]
//   wide    the shortcut, which the sum overwrites in place         [TM][Co]
//
// What moves through memory is the patch, the shortcut, the block's output (both contiguous:
// whole pixels), the last layer's output, and the weights.  Those come straight into registers:
// they were laid out beforehand in the order a wave consumes them (mxq_pack_block_weights: 1 KB
// per 32 x 32 MFMA operand), so a load is one contiguous KB, no LDS ring and no barrier stands
// between a wave and its next operand, and five barriers per tile are all that is left.  A CU
// takes in 64 bytes of weights per clock and multiplies them with the 64 pixels in the same time,
// which is why TM is no smaller where the tiles fill the chip.
//
// Rows in LDS are an odd number of 16-byte chunks apart: 16 consecutive rows' fragments hit
// distinct bank groups without a permutation, for any channel count.
//
// What bounds it: instruction issue.  Vector instructions and MFMAs, which overlap little (the waves
// of a work-group run in step from each barrier on), take 80 % of a CU's busy clocks in 56 x 56 x 64 and
// 66 % in 28 x 28 x 128 and 14 x 14 x 256 (counters, batch 64); the sum alone is 7 vector instructions
// per output of 64 ... 256 channels in the middle times four.  So what is not arithmetic has as few as
// possible: a weight's place is a scalar offset and an immediate, the three taps of a row are immediates
// where the channels are those of a kernel instance (KSB), the places of a tile's pixels in the tensors
// come from a table, and pieces of rows are walked by carries, not divided (947 -> 822 vector instructions
// a wave of 56 x 56 x 64, 1007 -> 892 and 2035 -> 1594 of the others); and a barrier waits for what it is for,
// not for weights or stores on their way.  The 3 x 3 layer of 256 channels takes in 590 KB of weights, 9200
// clocks at the 64 bytes a clock of a CU and as many as its products.  Measured in a quantized
// ResNet-50's pass at batch 64, before and after: 45.0 -> 39.9 us for 56 x 56 x 64 -> 256 -> 64, 33.9 ->
// 32.2 for 28 x 28 x 128, 26.6 -> 25.0 for 14 x 14 x 256; the pass's kernels 629 -> 603, one image's 210 ->
// 204.  Channels that no instance is made for, the block alone: 56 x 56 x 48 -> 192 -> 48 38.3 -> 37.7, 28
// x 28 x 96 -> 384 -> 96 31.5 -> 30.1, 14 x 14 x 192 -> 768 -> 192 18.5 -> 17.1.  As three launches, alone: 67,
// 53 and 43 us against 49, 30 and 28.
// Measured and not kept: the 3 x 3 layer's reduction shared by the waves that have no column tile of
// it (up to 128 channels in the middle half of them), or by 16 waves: level or behind, for the sums
// that are exchanged cost more vector instructions than the idle waves did time;
// a column tile's products made while the one before is finished (level, 100
// registers more), the second layer's operand held in registers (level), wave priorities (level).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"
#include "mxq_forms.h"
#include "mxq_gemm.h"

namespace mxq {
namespace {

// a lambda that is called rather than inlined would keep what it captures in scratch memory
#define MXQ_INLINE __attribute__((always_inline))

constexpr int kBlockLds = 160 * 1024;
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// The short forms of mxq_forms.h, and for the sum
//   fma(level, 2ta, fma(residual, 2tb, c)) as the form with the relu.  Both operands are small
//   integers in 16 bits, which read as half floats are that many times 2^-24: v_fma_mix_f32 takes
//   them as they are, without a conversion
// 7 instructions per output instead of 13.75.
struct SumForm {
  float ta, tb, c;  // for levels and residuals + 128, times 2^-24
};
__host__ __device__ inline SumForm sum_form(float ta, float tb) {  // ta, tb doubled
  return SumForm{ta * 16777216.0f, tb * 16777216.0f, 0.5f - 128.0f * (ta + tb)};
}
__device__ __forceinline__ float half_of(uint32_t w, int k) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return static_cast<float>(__builtin_bit_cast(h2, w)[k]);
}
__device__ __forceinline__ uint32_t short_sum4(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3,
                                               uint32_t y, const SumForm& f) {
  const uint32_t a[4] = {a0, a1, a2, a3};
  y ^= 0x80808080u;
  const uint32_t b[2] = {__builtin_amdgcn_perm(0u, y, 0x0c010c00u),
                         __builtin_amdgcn_perm(0u, y, 0x0c030c02u)};
  uint32_t w = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    w = __builtin_amdgcn_cvt_pk_u8_f32(
        __builtin_fmaf(half_of(a[k], 0), f.ta, __builtin_fmaf(half_of(b[k >> 1], k & 1), f.tb, f.c)),
        k, w);
  return halve4(w);
}

// What a launch needs to know of its three layers' scales and of the sum, prepared once
// (mxq_prepare_block).
struct BlockForms {
  EpiScalars s[3];
  RequantRule rule;
  float t[3], c[3];  // factor and constant of the layers' short forms
  SumForm sum;
  int has;       // bit i: layer i has one; bit 3: the sum has
  unsigned long long failed;  // of the tried pairs of factors
};
constexpr size_t kBlockForms = 192;
static_assert(sizeof(BlockForms) <= kBlockForms, "room for the forms");

struct BlockArgs {
  const int8_t* data;     // [N][H][W][C]
  const int8_t* weights;  // fragments of the three layers, one behind the other
  const BlockForms* forms;
  const char* prepared[3];  // the layers' int32 bias, kPreparedBias bytes in
  const int8_t* res;      // [M][Co]
  int8_t* out;            // [M][Co]
  int8_t* next;           // [M][Ca]
  int N, H, W, C, Cm, Co, Ca;
  int kb, ksb;            // MFMA steps of the 3 x 3 layer, and of one tap of it
  int ka;                 // ... of the last layer
  int at_c, at_a, kb_all; // where the second and third layer's fragments begin (KB), and all end
  int run;                // whether tiles are runs of pixels; else of tn images, th rows, tw columns
  int tn, th, tw, tiles_h, tiles_w;  // tiles down and across an image
  int area, across, count, rows;     // (above) and pixels of a tile, rows of its patch
  int off_patch, off_bias, off_table, off_pixel;  // bytes in LDS
  // what NW * 64 pieces are in rows and pieces beyond them, of the shortcut's slots and of the outputs
  int res_rows, res_rest, wide_rows, wide_rest, next_rows, next_rest;
  int parts, row_pitch;   // load instructions and bytes per row of the patch
  uint32_t magic_tiles_w, magic_tiles_h, magic_area, magic_across, magic_h2, magic_pixel,
      magic_res, magic_wide, magic_next, magic_tap;
  int relu_b, relu_a, tiles;
};

__host__ __device__ constexpr int odd(int chunks) { return chunks | 1; }
// ... of rows that are written in whole column tiles of 32 channels
__host__ __device__ constexpr int odd_tiles(int chunks) { return ((chunks + 1) & ~1) | 1; }

// A lane's pieces of rows that leave the launch: `chunks` pieces a row, rows `pitch` pieces apart in LDS
// from `at` on; the next one is `rows` rows and `rest` pieces further.
struct Pieces {
  int row, j, from;
  __host__ __device__ void begin(int first_row, int first_j, int at, int pitch) {
    row = first_row;
    j = first_j;
    from = at + (row * pitch + j) * 16;
  }
  __host__ __device__ void next(int rows, int rest, int chunks, int pitch) {
    row += rows;
    j += rest;
    from += (rows * pitch + rest) * 16;
    const bool carry = j >= chunks;
    j -= carry ? chunks : 0;
    row += carry;
    from += carry ? (pitch - chunks) * 16 : 0;
  }
  // what is read of LDS: where the lanes are more than the pieces, no more than there is of it
  __host__ __device__ int place(int tile_rows, int at) const { return row < tile_rows ? from : at; }
};
// From a row of the patch to the one below it, for the taps in row `row` of three.  The last of them
// has none below; what is read ahead there is not used.
__host__ __device__ inline int row_below(int row, int row_pitch) { return row < 2 ? row_pitch : 0; }

// floor(n / d) for n * d < 2^30, magic = 2^31 / d + 1: (2n + 1) / 2d is never an integer, and no
// case (d = 1) needs a branch, behind which the compiler would load the next argument
__device__ __forceinline__ int quotient(int n, uint32_t magic) {
  return static_cast<int>(__umulhi(2u * static_cast<uint32_t>(n) + 1u, magic));
}
// floor(n / d) for any 0 <= n < 2^31: the product above is at most one too large there
__device__ __forceinline__ int quotient_any(int n, int d, uint32_t magic) {
  const int q = quotient(n, magic);
  return q - (static_cast<uint32_t>(q) * static_cast<uint32_t>(d) > static_cast<uint32_t>(n));
}
uint32_t magic_of(int d) { return static_cast<uint32_t>((1ULL << 31) / static_cast<unsigned>(d) + 1); }

// WM x WN waves, each RT row tiles of 32 pixels by one column tile of 32 channels at a time.
// GB, GC: MFMA steps whose weights a wave requests together (the 3 x 3 layer's, and the whole
// reduction of the second layer).
// KSB: MFMA steps of a tap where the data has exactly 32 * KSB channels, so that the places of three
// taps in a row are constants; 0 for any other count, where a table in LDS has them.
// `tile` is one of p.tiles; or, of runs, the one that begins at pixel `first`.
template <int WM, int WN, int RT, int GB, int GC, int KSB>
__device__ __forceinline__ void block_tile(const BlockArgs& p, int tile, int first) {
  constexpr int NW = WM * WN, TM = 32 * WM * RT, GA = 8;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // every argument at once: left alone the compiler loads each of them where it is first used, a
  // round trip at a time, 3000 clocks before the first pixels are requested
  asm volatile("" ::"s"(p.data), "s"(p.weights), "s"(p.forms), "s"(p.prepared[0]),
               "s"(p.prepared[1]), "s"(p.prepared[2]), "s"(p.res), "s"(p.N), "s"(p.H), "s"(p.W),
               "s"(p.C), "s"(p.Cm), "s"(p.Co), "s"(p.Ca), "s"(p.kb), "s"(p.ksb),
               "s"(p.at_c), "s"(p.kb_all), "s"(p.off_patch), "s"(p.off_bias), "s"(p.off_table),
               "s"(p.run), "s"(p.area), "s"(p.across), "s"(p.count), "s"(p.rows), "s"(p.off_pixel),
               "s"(p.magic_area), "s"(p.magic_across), "s"(p.magic_h2),
               "s"(p.magic_pixel), "s"(p.parts), "s"(p.row_pitch), "s"(p.magic_res),
               "s"(p.magic_tap), "s"(p.tiles), "s"(p.res_rows), "s"(p.res_rest));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  // The tile's pixel i is pixel (h0, w0) + place start + i of rows of `across` in images of `area`
  // pixels, from image n0 on: a rectangle, whole images, or a run of pixels in the tensor's order.
  int n0, h0 = 0, w0 = 0, start_at = 0;
  if (p.run) {
    n0 = quotient_any(first, p.area, p.magic_area);
    start_at = first - n0 * p.area;
  } else {
    const int down = quotient(tile, p.magic_tiles_w), batch = quotient(down, p.magic_tiles_h);
    n0 = batch * p.tn;
    h0 = (down - batch * p.tiles_h) * p.th;
    w0 = (tile - down * p.tiles_w) * p.tw;
  }
  // rows of the patch are rows of the images one below the other, each with one more above and below
  const int H2 = p.H + 2, v0 = n0 * H2 + h0 + quotient(start_at, p.magic_across);
  const int CH = p.C >> 4, PP = odd(CH);
  const int row_pitch = p.row_pitch;  // bytes of a patch row
  const int PM = odd_tiles(p.Cm >> 4), CO = p.Co >> 4, PO = odd_tiles(CO);
  const int CA = p.Ca >> 4, PA = odd_tiles(CA);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  // 64 pieces of 16 bytes to `to` and on in LDS
  auto fetch = [&](int to, uint32_t from, v4i rsrc) MXQ_INLINE {
    dma_buffer(__builtin_amdgcn_readfirstlane(lds0 + to), from, rsrc);
  };

  const auto weights = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.weights), 0,
                                                         p.kb_all * 1024, 0x00020000);
  // Fragments number from ... from + G - 1, one at a time: a scalar offset and an immediate each, no
  // vector instruction.  Where there are none, zeros, and nothing is fetched: the lane's place is past
  // the end then, and the scalar part 0 (a buffer's bound is compared with the place alone, after the
  // scalar part was subtracted from it).
  const int lane16 = lane * 16;
  struct Fragments {
    int from, at;
  };
  auto fragments = [&](bool some, int from) MXQ_INLINE {
    return Fragments{some ? from : 0, some ? lane16 : 0x40000000};
  };
  auto fragment = [&](const Fragments& f, int i) MXQ_INLINE {
    return __builtin_bit_cast(v4i,
                              __builtin_amdgcn_raw_buffer_load_b128(
                                  weights, f.at + (i & 3) * 1024, (f.from + (i & ~3)) * 1024, 0));
  };
  auto load_first = [&](auto& w, const Fragments& f) MXQ_INLINE {
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(w) / sizeof(v4i)); ++i) w[i] = fragment(f, i);
  };
  const int tiles_b = (p.Cm + 31) >> 5, tiles_c = (p.Co + 31) >> 5, tiles_a = (p.Ca + 31) >> 5;
  const bool has_b = wn < tiles_b;
  v4i wb[GB];
  const int first_b = (has_b ? wn : 0) * p.kb;
  load_first(wb, fragments(true, first_b));

  // the patch: the tile's rows of every one of its images and one above and below, a column on
  // either side; zeros where they leave the image
  {
    const v4i rsrc = make_rsrc(p.data, static_cast<uint32_t>(p.N) * p.H * p.W * p.C);
    // A row of the patch is a whole number of load instructions, and a row is one scalar offset: the
    // lanes look at a row each, all at once, and what they find is read from them row by row; a lane's
    // place in a row moves on by carries from part to part.  Parts start at the wave behind the one that
    // took the last row of the part before, so that all take as many.  (The waves have little else to do
    // here, so each of the 55 instructions that looking at the row for every load takes is waited for.)  No
    // short circuits: a branch takes longer than what it skips.
    const int row_bytes = p.W * p.C;
    const int px_step = quotient(64, p.magic_pixel), j_rest = 64 - px_step * PP;
    for (int first_row = 0; first_row < p.rows; first_row += 64) {
      uint32_t row_at, row_none;
      {
        const int v = v0 + first_row + lane, n = quotient_any(v, H2, p.magic_h2), ih = v - n * H2 - 1;
        const int none = (n >= p.N) | (static_cast<unsigned>(ih) >= static_cast<unsigned>(p.H));
        row_at = static_cast<uint32_t>((n * p.H + ih) * row_bytes);
        row_none = static_cast<uint32_t>(none) << 31;
      }
      const int rows = p.rows - first_row < 64 ? p.rows - first_row : 64;
      int px = quotient(lane, p.magic_pixel), j = lane - px * PP, before = 0;
      for (int part = 0; part < p.parts; ++part) {
        const int iw = w0 + px - 1;
        const int none = (j >= CH) | (px >= p.across + 2) |
                         (static_cast<unsigned>(iw) >= static_cast<unsigned>(p.W));
        const uint32_t at = static_cast<uint32_t>(__mul24(iw, p.C) + 16 * j);
        const uint32_t outside = static_cast<uint32_t>(none) << 31;
        for (int r = (wave - before) & (NW - 1); r < rows; r += NW)
          fetch(p.off_patch + (first_row + r) * row_pitch + part * 1024,
                (at + __builtin_amdgcn_readlane(row_at, r)) |
                    (outside | __builtin_amdgcn_readlane(row_none, r)),
                rsrc);
        before += rows;
        j += j_rest;
        px += px_step;
        const int carry = j >= PP;
        j -= carry ? PP : 0;
        px += carry;
      }
    }
  }
  // For each of the tile's pixels where it lies in the wide tensors and in the last layer's result,
  // past their ends for those past the edges, and where the patch has its first tap.  With more than
  // 128 channels in the middle LDS has no room for three tables where it had for one (7 x 7 x 128 -> 256
  // -> 2048 -> 256 is 352 bytes short): every wave finds its own rows' first taps, while the patch is on
  // its way, and the last layer's places take those of the first one's bias, behind that layer.
  constexpr bool kOneTable = GC == 8;
  uint32_t* const wide_of = reinterpret_cast<uint32_t*>(smem + p.off_pixel);
  uint32_t* const next_of =
      kOneTable ? reinterpret_cast<uint32_t*>(smem + p.off_bias) : wide_of + TM;
  int* const place_of = reinterpret_cast<int*>(wide_of + 2 * TM);
  struct Pixel {
    int n, h, w, tx;
  };
  auto pixel_at = [&](int row) MXQ_INLINE {
    // rows without a pixel read the first one's; never stored
    const int i = start_at + (row < p.count ? row : 0);
    const int img = quotient_any(i, p.area, p.magic_area), rem = i - img * p.area;
    const int ty = quotient(rem, p.magic_across), tx = rem - ty * p.across;
    return Pixel{n0 + img, h0 + ty, w0 + tx, tx};
  };
  auto place_at = [&](const Pixel& x) MXQ_INLINE {
    return (x.n * H2 + x.h - v0) * row_pitch + x.tx * PP * 16;
  };
  static_assert(TM <= 64, "one wave makes the tables");
  const bool makes_tables = wave == NW - 1 && lane < TM;  // the wave that has least to fetch
  uint32_t next_at = kOutOfRange;
  if (makes_tables) {
    const Pixel x = pixel_at(lane);
    const bool ok = lane < p.count && x.n < p.N && x.h < p.H && x.w < p.W;
    const uint32_t pixel = static_cast<uint32_t>((x.n * p.H + x.h) * p.W + x.w);
    wide_of[lane] = ok ? pixel * p.Co : kOutOfRange;
    next_at = ok ? pixel * p.Ca : kOutOfRange;
    if constexpr (!kOneTable) {
      next_of[lane] = next_at;
      place_of[lane] = place_at(x);
    }
  }
  const int* const sbias = reinterpret_cast<const int*>(smem + p.off_bias);
  const int bias_c = (p.Cm + 31) & ~31, bias_a = bias_c + ((p.Co + 31) & ~31);
  // Whole column tiles of a layer's bias, zeros behind its last column: those of the 3 x 3 layer now,
  // the others' while that one runs.
  auto fetch_bias = [&](const char* prepared, int columns, int at, int i) MXQ_INLINE {
    const v4i rsrc = make_rsrc(prepared + kPreparedBias, 4u * columns);
    if (i * 256 + lane * 4 < ((columns + 31) & ~31))
      fetch(p.off_bias + at * 4 + i * 1024, i * 1024 + lane16, rsrc);
  };
  if (wave == 0) fetch_bias(p.prepared[0], p.Cm, 0, 0);  // no more than 256
  auto fetch_later_bias = [&]() MXQ_INLINE {
    const int n_c = (p.Co + 255) >> 8, n_a = (p.Ca + 255) >> 8;
    for (int it = NW - 1 - wave; it < n_c + n_a; it += NW) {
      const bool c = it < n_c;
      fetch_bias(c ? p.prepared[1] : p.prepared[2], c ? p.Co : p.Ca, c ? bias_c : bias_a,
                 c ? it : it - n_c);
    }
  };
  const EpiScalars s_b = p.forms->s[0], s_c = p.forms->s[1], s_a = p.forms->s[2];
  const RequantRule rule = p.forms->rule;
  const float t_b = p.forms->t[0], t_c = p.forms->t[1], t_a = p.forms->t[2];
  const float c_b = p.forms->c[0], c_a = p.forms->c[2];
  const SumForm form = p.forms->sum;
  const int has = p.forms->has;
  // where step k of the 3 x 3 layer reads, from the pixel's place under the first tap; steps behind
  // the last one have zero weights
  if constexpr (KSB == 0) {
    for (int k = tid; k < p.kb + 2 * GB; k += 64 * NW) {
      const int last = 9 * p.ksb - 1, at = k < last ? k : last;
      const int tap = quotient(at, p.magic_tap), kh = tap / 3;
      reinterpret_cast<int*>(smem + p.off_table)[k] =
          kh * row_pitch + (tap - 3 * kh) * PP * 16 + (at - tap * p.ksb) * 32;
    }
  }
  // The shortcut, a share of it at a time while the 3 x 3 layer runs.
  const v4i res_rsrc = make_rsrc(p.res, static_cast<uint32_t>(p.N) * p.H * p.W * p.Co);
  const int res_slots = TM * PO;
  int res_at = wave;
  int res_row = quotient(res_at * 64 + lane, p.magic_res);
  int res_j = res_at * 64 + lane - res_row * PO;
  auto fetch_shortcut = [&]() MXQ_INLINE {
    if (res_at * 64 < res_slots) {
      // (the pad of a row gets what follows the row in memory; tiles of 32 do not end on a whole load
      // instruction, and get their last row again behind it)
      const int row = TM % 64 == 0 || res_row < TM ? res_row : TM - 1;
      fetch(res_at * 1024, wide_of[row] + 16 * res_j, res_rsrc);
      res_at += NW;
      res_row += p.res_rows;
      res_j += p.res_rest;
      const bool carry = res_j >= PO;
      res_j -= carry ? PO : 0;
      res_row += carry;
    }
  };

  // this lane's rows: where they begin in each of the three
  const int frow = lane & 31, fgrp = lane >> 5;
  const int row0 = wm * RT * 32 + frow;
  int in_patch[RT];
  if constexpr (kOneTable) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      in_patch[rt] = p.off_patch + place_at(pixel_at(row0 + 32 * rt)) + fgrp * 16;
  }
  v16i acc[RT];
  // The bias as first accumulators.  Each row tile reads its own: registers are copied with vector
  // instructions, which this kernel is short of, so the compiler must not see that they are the same.
  auto start = [&](v16i (&acc)[RT], const int* bias) MXQ_INLINE {
    int at = static_cast<int>(reinterpret_cast<uintptr_t>(bias + 4 * fgrp));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      asm volatile("" : "+v"(at));
      const auto b = reinterpret_cast<const __attribute__((address_space(3))) v4i*>(at);
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const v4i x = b[2 * vq];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][4 * vq + i] = x[i];
      }
    }
  };
  // One group of G steps.  The pixels of a step are read kAhead steps before they are multiplied,
  // and a step's weights make room for those of the same step of the next group (fragments from
  // `from` on) as soon as they are used: G KB per wave are always on their way.  Requested all at
  // once, at the start of a group, the CU's 64 KB arrive in 1024 clocks and a latency, which is 1700
  // of the 1024 that eight steps should take.  The order is pinned: left alone the compiler sinks
  // the requests to the end of the group and reads each step's pixels right in front of its MFMAs.
  constexpr int kRing = NW * RT >= 16 && GC == 8 ? 4 : 2, kAhead = kRing - 1;
  v4i px[kRing][RT];
  auto read_pixels = [&](v4i (&x)[RT], const int (&base)[RT], int offset) MXQ_INLINE {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      x[rt] = *reinterpret_cast<const v4i*>(smem + base[rt] + offset);
  };
  // read(i, x): the pixels of step i of the group, for i up to G + kAhead - 1
  auto first_pixels = [&](auto read) MXQ_INLINE {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) read(i, px[i]);
  };
  auto multiply = [&](v16i (&acc)[RT], v4i w, const v4i (&x)[RT]) MXQ_INLINE {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      acc[rt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x[rt], acc[rt], 0, 0, 0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) asm volatile("" : "+v"(acc[rt]));
  };
  auto run_group = [&](auto& w, const Fragments& f, auto read) MXQ_INLINE {
    constexpr int G = sizeof(w) / sizeof(v4i);
    static_assert(G % kRing == 0, "the sets of pixels take turns");
#pragma unroll
    for (int i = 0; i < G; ++i) {
      read(i + kAhead, px[(i + kAhead) % kRing]);
      multiply(acc, w[i], px[i % kRing]);
      w[i] = fragment(f, i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // What this wave wrote to LDS, and what it had written there but for the newest `pending` loads, to
  // all of them.  Only what the barrier is for is waited for: weights on their way to registers, or
  // stores, at a barrier that publishes a result would cost a round trip to memory each.
  auto publish = [&](auto pending) MXQ_INLINE {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(pending)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto publish_written = [&]() MXQ_INLINE {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  publish(std::integral_constant<int, 0>());  // the patch, the bias, the tables

  // ---- 3 x 3 ------------------------------------------------------------------------------
  const int groups = p.kb / GB;
  if (has_b) {
    if constexpr (!kOneTable) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        in_patch[rt] = p.off_patch + place_of[row0 + 32 * rt] + fgrp * 16;
    }
    start(acc, sbias + 32 * wn);
    if constexpr (KSB != 0) {
      constexpr int kRow = 3 * KSB, kTap = odd(2 * KSB) * 16;
      static_assert(kRow % GB == 0, "a row of taps is whole groups");
      int below[RT];
      // step i of the taps in a row, or of the row below
      auto read = [&](int i, v4i (&x)[RT]) MXQ_INLINE {
        const int k = i < kRow ? i : i - kRow;
        read_pixels(x, i < kRow ? in_patch : below, k / KSB * kTap + k % KSB * 32);
      };
      first_pixels(read);
      for (int row = 0; row < 3; ++row) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) below[rt] = in_patch[rt] + row_below(row, row_pitch);
#pragma unroll
        for (int g = 0; g < kRow / GB; ++g) {
          fetch_shortcut();
          // (the last of them a latency ahead of the barrier behind the layer)
          if constexpr (GC == 8) fetch_shortcut();
          if (g == 0 && row == 1) fetch_later_bias();
          run_group(wb,
                    fragments(row < 2 || g + 1 < kRow / GB, first_b + row * kRow + (g + 1) * GB),
                    [&](int i, v4i (&x)[RT]) MXQ_INLINE { read(g * GB + i, x); });
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) in_patch[rt] = below[rt];
      }
    } else {
      // A group's places come with one read, a lane each, that is on its way while a group is multiplied
      // (pair by pair behind it, waited for each time: 10 x 10 x 1232 -> 112 25.7 us, 22.0 when all were
      // asked for at once, 20.6 so).
      const int* table =
          reinterpret_cast<const int*>(smem + p.off_table) + (lane < GB ? lane : 0);
      auto take_offsets = [&](int x, int (&o)[GB]) MXQ_INLINE {
#pragma unroll
        for (int i = 0; i < GB; ++i) o[i] = __builtin_amdgcn_readlane(x, i);
      };
      int now[GB], later[GB];
      take_offsets(table[0], now);
      take_offsets(table[GB], later);
      auto read = [&](int i, v4i (&x)[RT]) MXQ_INLINE {
        read_pixels(x, in_patch, i < GB ? now[i] : later[i - GB]);
      };
      first_pixels(read);
      for (int g = 0; g < groups; ++g) {
        fetch_shortcut();
        if (g == 0) fetch_later_bias();
        const int ahead = table[2 * GB];
        table += GB;
        run_group(wb, fragments(g + 1 < groups, first_b + (g + 1) * GB), read);
#pragma unroll
        for (int i = 0; i < GB; ++i) now[i] = later[i];
        take_offsets(ahead, later);
      }
    }
  } else {
    fetch_later_bias();
  }
  while (res_at * 64 < res_slots) fetch_shortcut();
  v4i wc[GC];
  load_first(wc, fragments(wn < tiles_c, p.at_c + wn * GC));
  // column tile t of a layer's int8 result into rows of `pitch` chunks at the patch's place
  auto finish = [&](int t, int pitch, auto pack) MXQ_INLINE {
#pragma unroll
    for (int vq = 0; vq < 4; ++vq)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        *reinterpret_cast<uint32_t*>(smem + p.off_patch + (row0 + 32 * rt) * pitch * 16 + 32 * t +
                                     8 * vq + 4 * fgrp) =
            pack(acc[rt][4 * vq], acc[rt][4 * vq + 1], acc[rt][4 * vq + 2], acc[rt][4 * vq + 3]);
  };
  auto finish_layer = [&](const EpiScalars s, const float factor, const float constant, bool has,
                          int relu, int t, int pitch) MXQ_INLINE {
    if (relu && has)
      finish(t, pitch,
             [&](int a, int b, int c, int d) { return short_relu4(a, b, c, d, factor, constant); });
    else if (relu)
      finish(t, pitch,
             [&](int a, int b, int c, int d) { return epi_requant_pack<true>(a, b, c, d, s); });
    else
      finish(t, pitch,
             [&](int a, int b, int c, int d) { return epi_requant_pack<false>(a, b, c, d, s); });
  };
  __builtin_amdgcn_s_barrier();  // every wave is through with the patch
  asm volatile("" ::: "memory");
  if (has_b) finish_layer(s_b, t_b, c_b, (has & 1) != 0, p.relu_b, wn, PM);
  if (kOneTable && makes_tables) next_of[lane] = next_at;
  publish(std::integral_constant<int, GC>());  // the result, and the shortcut in front of `wc`

  // ---- 1 x 1 and the sum ------------------------------------------------------------------
  // where this lane's rows are read as an operand, and where its outputs of a column tile lie
  int in_mid[RT], in_wide[RT], at_wide[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    in_mid[rt] = p.off_patch + (row0 + 32 * rt) * PM * 16 + fgrp * 16;
    in_wide[rt] = (row0 + 32 * rt) * PO * 16 + fgrp * 16;
    at_wide[rt] = (row0 + 32 * rt) * PO * 16 + fgrp * 4;
  }
  auto widen = [&](auto how) MXQ_INLINE {
    constexpr int F = decltype(how)::value;
    for (int t = wn; t < tiles_c; t += WN) {
      const Fragments f = fragments(t + WN < tiles_c, p.at_c + (t + WN) * GC);
      uint32_t shortcut[RT][4];
      start(acc, sbias + bias_c + 32 * t);
      read_pixels(px[0], in_mid, 0);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
          shortcut[rt][vq] =
              *reinterpret_cast<const uint32_t*>(smem + at_wide[rt] + 32 * t + 8 * vq);
#pragma unroll
      for (int i = 0; i < GC; ++i) {
        if (i + 1 < GC) read_pixels(px[(i + 1) & 1], in_mid, 32 * (i + 1));
        multiply(acc, wc[i], px[i & 1]);
        wc[i] = fragment(f, i);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int vq = 0; vq < 4; ++vq)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const int a = acc[rt][4 * vq], b = acc[rt][4 * vq + 1], c = acc[rt][4 * vq + 2],
                    d = acc[rt][4 * vq + 3];
          const uint32_t y = shortcut[rt][vq];
          uint32_t w;
          if constexpr (F == 2) {
            w = short_sum4(short_level(a, t_c), short_level(b, t_c), short_level(c, t_c),
                           short_level(d, t_c), y, form);
          } else {
            const uint32_t x = epi_requant_pack<false>(a, b, c, d, s_c);
            w = F == 1 ? sum_requant4<true>(x, y, rule) : sum_requant4_general<true>(x, y, rule);
          }
          *reinterpret_cast<uint32_t*>(smem + at_wide[rt] + 32 * t + 8 * vq) = w;
        }
    }
  };
  if ((has & 10) == 10)
    widen(std::integral_constant<int, 2>());
  else if (rule.fast)
    widen(std::integral_constant<int, 1>());
  else
    widen(std::integral_constant<int, 0>());
  v4i wa[GA];
  if (p.Ca != 0) load_first(wa, fragments(wn < tiles_a, p.at_a + wn * p.ka));
  publish_written();

  // Rows of `chunks` pieces, `pitch` apart in LDS, to their pixels.  No streaming stores: the
  // next block reads both outputs, and what it finds in the memory-side cache it does not fetch from
  // memory (quantized ResNet-50 at batch 64, all blocks with streaming stores 5 % behind plain ones;
  // written through, kDeviceScope, a block is 1.5 to 2.3 us ahead of those, which leave up to 32 MB of
  // dirty lines to the launch's end).
  auto leave = [&](int at, int chunks, int pitch, uint32_t magic, int rows, int rest,
                   const uint32_t* pixel_of, int8_t* out) MXQ_INLINE {
    const auto to = __builtin_amdgcn_make_buffer_rsrc(
        out, 0, static_cast<uint32_t>(p.N) * p.H * p.W * chunks * 16, 0x00020000);
    Pieces piece;
    const int first = quotient(tid, magic);
    piece.begin(first, tid - first * chunks, at, pitch);
    for (int left = TM * chunks; left > 0; left -= 64 * NW) {
      // (rows past the tile's are written nowhere)
      const uint32_t pixel = piece.row < TM ? pixel_of[piece.row] : kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b128(
          __builtin_bit_cast(v4u, *reinterpret_cast<const v4i*>(smem + piece.place(TM, at))), to,
          pixel + 16 * piece.j, 0, kDeviceScope);
      piece.next(rows, rest, chunks, pitch);
    }
  };
  leave(0, CO, PO, p.magic_wide, p.wide_rows, p.wide_rest, wide_of, p.out);
  if (p.Ca == 0) return;

  // ---- the next block's first 1 x 1 ---------------------------------------------------------
  const int groups_a = p.ka / GA;
  for (int t = wn; t < tiles_a; t += WN) {
    start(acc, sbias + bias_a + 32 * t);
    first_pixels([&](int i, v4i (&x)[RT]) MXQ_INLINE { read_pixels(x, in_wide, 32 * i); });
    int at[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) at[rt] = in_wide[rt];
    for (int g = 0; g < groups_a; ++g) {
      const bool last = g + 1 == groups_a;
      run_group(wa,
                fragments(!last || t + WN < tiles_a,
                          p.at_a + (last ? (t + WN) * p.ka : t * p.ka + (g + 1) * GA)),
                [&](int i, v4i (&x)[RT]) MXQ_INLINE { read_pixels(x, at, 32 * i); });
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) at[rt] += 32 * GA;
    }
    finish_layer(s_a, t_a, c_a, (has & 4) != 0, p.relu_a, t, PA);
  }
  publish_written();
  leave(p.off_patch, CA, PA, p.magic_next, p.next_rows, p.next_rest, next_of, p.next);
}

template <int WM, int WN, int RT, int GB, int GC, int KSB>
__global__ __launch_bounds__(64 * WM * WN, GC < 8 ? 4 : 2) void block_kernel(BlockArgs p) {
  // an XCD takes a run of neighbouring tiles: they share halo rows in its L2
  const int per = (p.tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile < p.tiles) block_tile<WM, WN, RT, GB, GC, KSB>(p, tile, tile * 32 * WM * RT);
}

// Runs of pixels: p.tiles (a multiple of 8) of 64 and the rest in halves behind them.
template <int GB, int GC, int KSB>
__global__ __launch_bounds__(512, GC < 8 ? 4 : 2) void block_halves_kernel(BlockArgs p) {
  const int block = blockIdx.x;
  if (block < p.tiles)
    block_tile<1, 8, 2, GB, GC, KSB>(p, 0, 64 * ((block & 7) * (p.tiles >> 3) + (block >> 3)));
  else
    block_tile<1, 8, 1, GB, GC, KSB>(p, 0, 64 * p.tiles + 32 * (block - p.tiles));
}

// [O][taps][C] rows -> fragments [ceil(O / 32)][steps][64 lanes][16 bytes]: lane l of step
// tap * per_tap + s holds bytes 32 * s + 16 * (l / 32) ... + 15 of tap `tap` of row l % 32 of the
// column tile, zeros where there are none.
__global__ __launch_bounds__(256) void pack_fragments_kernel(const v4i* in, v4i* out, int O,
                                                             int taps, int chunks, int per_tap,
                                                             int steps, unsigned pieces) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const int lane = i & 63;
  const unsigned f = i >> 6;
  const int t = f / steps, k = f - t * steps;
  const int tap = k / per_tap, c = 2 * (k - tap * per_tap) + (lane >> 5);
  const int n = 32 * t + (lane & 31);
  const bool ok = n < O && tap < taps && c < chunks;
  out[i] = ok ? in[(static_cast<size_t>(n) * taps + tap) * chunks + c] : v4i{0, 0, 0, 0};
}

// The search for the forms, in three launches: nothing found yet; work-groups 0 ... 2 each look for
// a layer's (layers 0 and 2 with the relu, 1 without), and the others take kShares to a pair of
// factors for the sum, each a share of the operands; then what those found.
struct PrepareArgs {
  const char* prepared[3];
  const float* res_min;
  const float* res_max;
  float layer_range, sum_min, sum_max;
  BlockForms* out;
};
constexpr int kPairs = 49, kShares = 8;
__device__ __forceinline__ RequantRule block_rule(const PrepareArgs& p) {
  return sum_requant_rule(dev_maxabs(-p.layer_range, p.layer_range),
                          dev_maxabs(*p.res_min, *p.res_max), p.sum_min, p.sum_max);
}
// doubled factors number c of the rule, where they can be used
__device__ __forceinline__ bool pair_of_factors(const RequantRule& r, int c, float* a, float* b) {
  const double level = 2.0 * static_cast<double>(r.in_scale) * static_cast<double>(r.qscale);
  const float ta = static_cast<float>(r.s0 * level), tb = static_cast<float>(r.s1 * level);
  *a = moved(ta, c % 7);
  *b = moved(tb, c / 7);
  return r.fast && ta > 1e-30f && tb > 1e-30f && ta < 1e30f && tb < 1e30f;
}
__global__ void clear_forms_kernel(BlockForms* out) {
  out->has = 0;
  out->failed = 0;
}
__global__ void finish_forms_kernel(PrepareArgs p) {
  BlockForms* const out = p.out;
  out->rule = block_rule(p);
  const int pair = __builtin_ctzll(~out->failed);  // the first that has not
  float a, b;
  const bool usable = pair_of_factors(out->rule, pair % kPairs, &a, &b);
  out->sum = sum_form(a, b);
  if (usable && pair < kPairs) out->has |= 8;
}
__global__ __launch_bounds__(1024) void prepare_block_kernel(PrepareArgs p) {
  const int tid = threadIdx.x;
  __shared__ FormSearch search;
  BlockForms* const out = p.out;
  if (blockIdx.x < 3) {
    const int layer = blockIdx.x;
    if (p.prepared[layer] == nullptr) return;
    const EpiScalars s = *reinterpret_cast<const EpiScalars*>(p.prepared[layer]);
    const LayerForm f = find_form(s, layer != 1, &search);
    if (tid == 0) {
      out->s[layer] = s;
      out->t[layer] = f.t;
      out->c[layer] = f.c;
      if (f.has) atomicOr(&out->has, 1 << layer);
    }
  } else {
    // a share of the operands' pairs each
    const RequantRule r = block_rule(p);
    const int pair = (blockIdx.x - 3) / kShares, share = (blockIdx.x - 3) % kShares;
    float a, b;
    if (!pair_of_factors(r, pair, &a, &b)) return;
    bool differs = false;
    for (int i = share * 1024 + tid; i < 64 * 256; i += 1024 * kShares) {
      const int a0 = 4 * (i >> 8) - 127, y0 = (i & 255) - 128;  // a0 ... a0 + 3
      int x[4];
      uint32_t packed = 0;
      for (int k = 0; k < 4; ++k) {
        x[k] = a0 + k < 127 ? a0 + k : 127;  // the last quad is one short
        packed |= (static_cast<uint32_t>(x[k]) & 0xffu) << (8 * k);
      }
      const uint32_t y = (static_cast<uint32_t>(y0) & 0xffu) * 0x01010101u;
      differs |= short_sum4(x[0] + 128, x[1] + 128, x[2] + 128, x[3] + 128, y, sum_form(a, b)) !=
                 sum_requant4_general<true>(packed, y, r);
    }
    if (__syncthreads_or(differs) != 0 && tid == 0) atomicOr(&out->failed, 1ULL << pair);
  }
}

int up(int n, int unit) { return (n + unit - 1) / unit * unit; }

// How a block of this shape is laid out; `tiles` is 0 where it does not fit.
struct BlockPlan {
  int variant = 0;  // 64, 128 or 256: the channels in the middle, at most
  int tm = 0, tiles = 0;
  int halves = 0;  // tiles of half the size behind them
  int steps[3] = {0, 0, 0};
  size_t fragments[3] = {0, 0, 0};  // KB
  int run = 0, tn = 1, th = 1, tw = 1, tiles_h = 1, tiles_w = 1, rows = 0;
  int parts = 0, row_pitch = 0, off_patch = 0, off_bias = 0, off_table = 0, off_pixel = 0, lds = 0;
};
// Tile and fragments of a block over these channels; false where no kernel takes them.
bool plan_layers(int C, int Cm, int Co, int Ca, BlockPlan* b) {
  for (int v : {C, Cm, Co})
    if (v <= 0 || v % 16 != 0 || v > 8192) return false;
  if (Ca < 0 || Ca % 16 != 0 || Ca > 8192 || Cm > 256) return false;
  b->variant = Cm <= 64 ? 64 : Cm <= 128 ? 128 : 256;
  b->tm = 64;
  b->steps[0] = up(9 * ((C + 31) / 32), b->variant == 256 ? 8 : 6);
  b->steps[1] = b->variant / 32;
  b->steps[2] = up((Co + 31) / 32, 8);
  const int columns[3] = {Cm, Co, Ca};
  size_t kb = 0;
  for (int i = 0; i < 3; ++i) {
    b->fragments[i] = static_cast<size_t>((columns[i] + 31) / 32) * b->steps[i];
    kb += b->fragments[i];
  }
  return kb < 0x100000;  // offsets in KB below 1 GiB
}
// The parts of LDS for a patch of b->rows rows of b->tw + 2 pixels; whether they fit.
bool fit_lds(BlockPlan* b, int C, int Cm, int Co, int Ca) {
  b->parts = up((b->tw + 2) * odd(C / 16), 64) / 64;
  // a row begins where the bank group of the pixel behind the last output pixel of the row before
  // it would be, so that 16 output pixels in a row hit distinct ones across the end of a row as well
  b->row_pitch = b->parts * 1024 + b->tw * odd(C / 16) % 16 * 16;
  const long long first = static_cast<long long>(b->rows) * b->row_pitch;
  if (first > kBlockLds) return false;
  // whole load instructions of the shortcut and of the bias; what a row's padded steps read past
  // the end of their part lies in the next one
  const int wide = up(b->tm * odd_tiles(Co / 16), 64) * 16;
  const int mid = b->tm * odd_tiles((Cm > Ca ? Cm : Ca) / 16) * 16;
  const int patch = first > mid ? static_cast<int>(first) : mid;
  const int bias = 4 * (up(Cm, 32) + up(Co, 32) + up(Ca, 32));
  const int table = 4 * (b->steps[0] + 2 * 8);
  const long long lds = static_cast<long long>(wide) + patch + bias + table +
                        4 * b->tm * (b->variant == 256 ? 1 : 3);
  b->off_patch = wide;
  b->off_bias = wide + patch;
  b->off_table = b->off_bias + bias;
  b->off_pixel = b->off_table + table;
  b->lds = static_cast<int>(lds);
  return lds <= kBlockLds;
}
BlockPlan plan_tiles(int N, int H, int W, int C, int Cm, int Co, int Ca, int tm) {
  BlockPlan b;
  if (!plan_layers(C, Cm, Co, Ca, &b)) return b;
  b.tm = tm;
  if (N <= 0 || H <= 0 || W <= 0 || W > 8192 || H > 8192) return b;
  const long long M = static_cast<long long>(N) * H * W;
  const long long widest = Co > C ? Co : C;
  if (M * (widest > Ca ? widest : Ca) >= (1LL << 31) || (M + 64) * 2 >= (1LL << 31) ||
      (static_cast<long long>(H) * W + 64) * W >= (1LL << 30) ||
      (N + 1LL) * (H + 2) + 256 >= (1LL << 30))
    return b;
  // A run of pixels in the tensor's order wastes no row of a tile, but its patch is three to five
  // times the tile: 36 KB for 64 pixels of a 56 x 56 plane over 64 channels where 8 x 8 of them need
  // 10, and LDS is what limits the work-groups a CU holds.  So runs where a CU holds one anyway or
  // where it still holds two; rectangles elsewhere.  (Batch 64, runs / rectangles: 56 x 56 x 64 63.1 /
  // 49.3 us, 30 x 30 x 64 20.7 / 19.2, 28 x 28 x 128 30.4 / 32.0, 17 x 17 x 128 13.9 / 16.1, 40 x 40 x 128, where
  // a CU does not hold two, 54.0 / 53.4, 14 x 14 x 256 27.6 / 29.5, 24 x 24 x 256 73.7 / 79.8.  On tiles of 32
  // rectangles are ahead by up to 5 %: 28 x 28 x 128 on one image 7.6 / 7.2.)
  if (b.variant > 64) {
    b.run = 1;
    // its rows, one above and below, two more for every image boundary inside
    b.rows = (b.tm + W - 2) / W + 1 + 2 + 2 * ((b.tm + H * W - 2) / (H * W));
    b.tw = W;
    const long long tiles = (M + b.tm - 1) / b.tm;
    if (fit_lds(&b, C, Cm, Co, Ca) && (b.variant == 256 || 2 * b.lds <= kBlockLds)) {
      b.tiles = static_cast<int>(tiles);
      return b;
    }
    b.run = 0;
  }
  // Whole images where one is no larger than a tile; else the rectangle that wastes least, a pixel
  // of the halo counted as a quarter of a row of the tile.
  if (H * W <= b.tm) {
    b.tn = b.tm / (H * W) < N ? b.tm / (H * W) : N;
    b.th = H;
    b.tw = W;
  } else {
    long long best = -1;
    for (int across = (W + b.tm - 1) / b.tm; across <= W; ++across) {
      const int tw = (W + across - 1) / across;
      if ((W + tw - 1) / tw != across) continue;
      const int most = b.tm / tw < H ? b.tm / tw : H, down = (H + most - 1) / most;
      const int th = (H + down - 1) / down;
      const long long cost = static_cast<long long>(across) * down * (4 * b.tm + (th + 2) * (tw + 2));
      if (best < 0 || cost < best) {
        best = cost;
        b.th = th;
        b.tw = tw;
        b.tiles_h = down;
        b.tiles_w = across;
      }
    }
  }
  b.rows = b.tn * (b.th + 2);
  const long long tiles = static_cast<long long>((N + b.tn - 1) / b.tn) * b.tiles_h * b.tiles_w;
  if (fit_lds(&b, C, Cm, Co, Ca) &&
      tiles * (b.tiles_w > b.tiles_h ? b.tiles_w : b.tiles_h) < (1 << 30))
    b.tiles = static_cast<int>(tiles);
  return b;
}

// Tiles of 64 pixels: a CU then multiplies a weight as long as it takes in the next one.  Where they
// would leave half of the CUs idle, of 32: a tile's chain is shorter by half of its products and its
// vector work (28 x 28 x 128 on one image 9.3 us -> 7.5, on 8 images 10.1 -> 8.4; 14 x 14 x 256 on
// 4 images 22.7 -> 16.9, on 32 24.4 -> 18.9; 56 x 56 x 64 on two, 98 tiles, 8.4 -> 6.7).  And where a few
// runs are left over when every CU has had as many, those go in halves, so that fewer CUs end with a
// whole tile more than the others (28 x 28 x 128 at batch 64, 784 tiles on 256 CUs, 30.8 -> 29.2; at batch
// 24 15.9 -> 14.4, at 32, 136 left over, 17.3 and 17.6).
BlockPlan plan_block(int N, int H, int W, int C, int Cm, int Co, int Ca) {
  BlockPlan b = plan_tiles(N, H, W, C, Cm, Co, Ca, 64);
  const int cus = num_cus(), over = b.tiles % cus;
  if (b.run && b.variant > 64 && b.tiles > cus && over != 0 && 2 * over <= cus && cus % 8 == 0) {
    b.tiles -= over;
    b.halves = static_cast<int>((static_cast<long long>(N) * H * W - 64LL * b.tiles + 31) / 32);
  }
  if (b.tiles == 0 || 2 * b.tiles > cus) return b;
  const BlockPlan half = plan_tiles(N, H, W, C, Cm, Co, Ca, 32);
  return half.tiles > 0 ? half : b;
}

template <int WM, int WN, int RT, int GB, int GC>
void launch_block(hipStream_t s, BlockArgs a, const BlockPlan& b) {
  constexpr int n = 64 * WM * WN, ksb = GC;  // as many channels in as in the middle
  const int pitch = odd_tiles(a.Co / 16);
  a.res_rows = n / pitch;
  a.res_rest = n % pitch;
  a.wide_rows = n / (a.Co / 16);
  a.wide_rest = n % (a.Co / 16);
  a.next_rows = a.Ca ? n / (a.Ca / 16) : 0;
  a.next_rest = a.Ca ? n % (a.Ca / 16) : 0;
  const bool known = a.C == 32 * ksb;
  if (b.halves != 0) {
    const dim3 grid(static_cast<unsigned>(b.tiles + b.halves));
    if constexpr (WM == 1 && WN == 8 && RT == 2) {
      if (known)
        hipLaunchKernelGGL((block_halves_kernel<GB, GC, ksb>), grid, dim3(n), b.lds, s, a);
      else
        hipLaunchKernelGGL((block_halves_kernel<GB, GC, 0>), grid, dim3(n), b.lds, s, a);
    }
  } else {
    const dim3 grid(static_cast<unsigned>((a.tiles + 7) / 8 * 8));
    if (known)
      hipLaunchKernelGGL((block_kernel<WM, WN, RT, GB, GC, ksb>), grid, dim3(n), b.lds, s, a);
    else
      hipLaunchKernelGGL((block_kernel<WM, WN, RT, GB, GC, 0>), grid, dim3(n), b.lds, s, a);
  }
  MXQ_LAUNCH_CHECK();
}

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" {

// Whether it is also the faster way.  It is from one image on with up to 128 channels in the middle
// (56 x 56 x 64: 6.5 us against 14.7 in three launches on one image, 49 against 67 on 64; 28 x 28 x 128 7.6
// / 15.0 and 30 / 53).  Above that a tile alone takes 16 us, most of it the 1.1 MB of weights that a CU
// takes in: 7 tiles (7 x 7 x 256 on 4 images) 16.2 us against 14.7, 13 tiles 16.5 against 16.1 ... 16.5, 25 tiles
// 16.8 against 19.4, 98 of 32 pixels 18.9 against 30.0, 196 of 64 27.6 against 42.7.  (The line was drawn
// where an earlier form of the kernel met the three launches; this one would already be ahead at 19
// tiles, 16.8 against 18.9.)
int mxq_quantized_block_fits(int N, int H, int W, int C, int C_mid, int C_out, int C_next) {
  try {
    const BlockPlan b = plan_block(N, H, W, C, C_mid, C_out, C_next);
    return b.tiles > 0 && (b.variant < 256 || b.tiles >= 20) ? 1 : 0;
  } catch (...) {  // no device to ask
    return 0;
  }
}

size_t mxq_quantized_block_weights(int C, int C_mid, int C_out, int C_next) {
  BlockPlan b;
  if (!plan_layers(C, C_mid, C_out, C_next, &b)) return 0;
  return 1024 * (b.fragments[0] + b.fragments[1] + b.fragments[2]);
}

int mxq_pack_block_weights(void* stream, const int8_t* first, const int8_t* second,
                           const int8_t* third, int C, int C_mid, int C_out, int C_next,
                           int8_t* out) {
  MXQ_API_BEGIN();
  BlockPlan b;
  MXQ_CHECK(plan_layers(C, C_mid, C_out, C_next, &b), "bad channel counts");
  const int8_t* const in[3] = {first, second, third};
  const int rows[3] = {C_mid, C_out, C_next}, columns[3] = {C, C_mid, C_out};
  MXQ_CHECK(out != nullptr && aligned16(out), "null or unaligned pointer");
  for (int i = 0; i < 3; ++i) {
    if (rows[i] == 0) continue;
    MXQ_CHECK(in[i] != nullptr && aligned16(in[i]), "null or unaligned pointer");
    const unsigned pieces = static_cast<unsigned>(b.fragments[i] * 64);
    hipLaunchKernelGGL(pack_fragments_kernel, dim3((pieces + 255) / 256), dim3(256), 0,
                       static_cast<hipStream_t>(stream), reinterpret_cast<const v4i*>(in[i]),
                       reinterpret_cast<v4i*>(out), rows[i], i == 0 ? 9 : 1, columns[i] / 16,
                       (columns[i] + 31) / 32, b.steps[i], pieces);
    MXQ_LAUNCH_CHECK();
    out += b.fragments[i] * 1024;
  }
  MXQ_API_END();
}

size_t mxq_quantized_block_forms(void) { return kBlockForms; }

int mxq_prepare_block(void* stream, const void* prepared_first, const void* prepared_second,
                      const void* prepared_third, const float* min_residual,
                      const float* max_residual, float min_calib, float max_calib,
                      float sum_min_calib, float sum_max_calib, void* forms) {
  MXQ_API_BEGIN();
  MXQ_CHECK(prepared_first && prepared_second && min_residual && max_residual && forms,
            "null pointer");
  for (const void* v : {prepared_first, prepared_second, prepared_third,
                        static_cast<const void*>(forms)})
    MXQ_CHECK(aligned16(v), "unaligned pointer");
  PrepareArgs a = {};
  a.prepared[0] = static_cast<const char*>(prepared_first);
  a.prepared[1] = static_cast<const char*>(prepared_second);
  a.prepared[2] = static_cast<const char*>(prepared_third);
  a.res_min = min_residual;
  a.res_max = max_residual;
  const float x = fabsf(min_calib), y = fabsf(max_calib);
  a.layer_range = (x < y) ? y : x;
  a.sum_min = sum_min_calib;
  a.sum_max = sum_max_calib;
  a.out = static_cast<BlockForms*>(forms);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(clear_forms_kernel, dim3(1), dim3(1), 0, s, a.out);
  MXQ_LAUNCH_CHECK();
  hipLaunchKernelGGL(prepare_block_kernel, dim3(3 + kPairs * kShares), dim3(1024), 0, s, a);
  MXQ_LAUNCH_CHECK();
  hipLaunchKernelGGL(finish_forms_kernel, dim3(1), dim3(1), 0, s, a);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

int mxq_quantized_block(void* stream, const int8_t* data, const int8_t* weights,
                        const void* forms, const void* prepared_first,
                        const void* prepared_second, const void* prepared_third, int N, int H,
                        int W, int C, int C_mid, int C_out, int C_next, const int8_t* residual,
                        int8_t* out, int8_t* next, int relu_first, int relu_third) {
  MXQ_API_BEGIN();
  const BlockPlan b = plan_block(N, H, W, C, C_mid, C_out, C_next);
  MXQ_CHECK(b.tiles > 0, "a block of this shape does not fit");
  MXQ_CHECK(data && weights && forms && residual && out && prepared_first && prepared_second &&
                (C_next == 0 || (next && prepared_third)),
            "null pointer");
  for (const void* v : {static_cast<const void*>(data), static_cast<const void*>(weights), forms,
                        prepared_first, prepared_second, prepared_third,
                        static_cast<const void*>(residual), static_cast<const void*>(out),
                        static_cast<const void*>(next)})
    MXQ_CHECK(aligned16(v), "unaligned pointer");
  BlockArgs a = {};
  a.data = data;
  a.weights = weights;
  a.forms = static_cast<const BlockForms*>(forms);
  a.prepared[0] = static_cast<const char*>(prepared_first);
  a.prepared[1] = static_cast<const char*>(prepared_second);
  a.prepared[2] = static_cast<const char*>(prepared_third);
  a.res = residual;
  a.out = out;
  a.next = next;
  a.N = N; a.H = H; a.W = W; a.C = C; a.Cm = C_mid; a.Co = C_out; a.Ca = C_next;
  
  a.kb = b.steps[0];
  a.ksb = (C + 31) / 32;
  a.ka = b.steps[2];
  a.at_c = static_cast<int>(b.fragments[0]);
  a.at_a = static_cast<int>(b.fragments[0] + b.fragments[1]);
  a.kb_all = static_cast<int>(a.at_a + b.fragments[2]);
  a.off_patch = b.off_patch;
  a.off_bias = b.off_bias;
  a.off_table = b.off_table;
  a.run = b.run; a.tn = b.tn; a.th = b.th; a.tw = b.tw; a.tiles_h = b.tiles_h; a.tiles_w = b.tiles_w;
  a.area = b.run ? H * W : b.th * b.tw;
  a.across = b.tw;
  a.count = b.run ? b.tm : b.tn * b.th * b.tw;
  a.rows = b.rows;
  a.off_pixel = b.off_pixel;
  a.magic_tiles_w = magic_of(b.tiles_w);
  a.magic_tiles_h = magic_of(b.tiles_h);
  a.magic_area = magic_of(a.area);
  a.magic_across = magic_of(b.tw);
  a.magic_h2 = magic_of(H + 2);
  a.magic_pixel = magic_of(odd(C / 16));
  a.parts = b.parts;
  a.row_pitch = b.row_pitch;
  a.magic_res = magic_of(odd_tiles(C_out / 16));
  a.magic_wide = magic_of(C_out / 16);
  a.magic_tap = magic_of(a.ksb);
  a.magic_next = C_next ? magic_of(C_next / 16) : 0;
  a.relu_b = relu_first != 0;
  a.relu_a = relu_third != 0;
  a.tiles = b.tiles;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (b.tm == 32) {
    if (b.variant == 64)
      launch_block<1, 4, 1, 6, 2>(s, a, b);
    else if (b.variant == 128)
      launch_block<1, 8, 1, 6, 4>(s, a, b);
    else
      launch_block<1, 8, 1, 8, 8>(s, a, b);
  } else if (b.variant == 64) {
    launch_block<2, 2, 1, 6, 2>(s, a, b);
  } else if (b.variant == 128) {
    launch_block<1, 8, 2, 6, 4>(s, a, b);
  } else {
    launch_block<1, 8, 2, 8, 8>(s, a, b);
  }
  MXQ_API_END();
}

#ifdef MXQ_TEST_HOOKS
// The bytes of LDS that a tile of `tile` pixels has, and how far the reads of the outputs' pieces, of
// the 1 x 1 layers' operands and of the constant taps reach.
int mxq_test_block_lds(int N, int H, int W, int C, int C_mid, int C_out, int C_next, int tile,
                       int* lds, int* reach) {
  MXQ_API_BEGIN();
  MXQ_CHECK((tile == 32 || tile == 64) && lds != nullptr && reach != nullptr, "bad arguments");
  *lds = *reach = 0;
  const BlockPlan b = plan_tiles(N, H, W, C, C_mid, C_out, C_next, tile);
  if (b.tiles == 0) return 0;
  *lds = b.lds;
  const int lanes = b.variant == 64 ? 256 : 512;
  auto read = [&](int place) { *reach = place + 16 > *reach ? place + 16 : *reach; };
  auto leave = [&](int at, int chunks) {
    const int pitch = odd_tiles(chunks);
    for (int tid = 0; tid < lanes && chunks != 0; ++tid) {
      Pieces piece;
      piece.begin(tid / chunks, tid % chunks, at, pitch);
      for (int left = tile * chunks; left > 0; left -= lanes) {
        read(piece.place(tile, at));
        piece.next(lanes / chunks, lanes % chunks, chunks, pitch);
      }
    }
  };
  leave(0, C_out / 16);
  leave(b.off_patch, C_next / 16);
  // the last row of each operand, whole steps and what is read ahead of them
  const int ahead = b.variant == 256 && tile == 64 ? 3 : 1;
  read(b.off_patch + (tile - 1) * odd_tiles(C_mid / 16) * 16 + 16 + 32 * (b.steps[1] - 1));
  if (C_next != 0)
    read((tile - 1) * odd_tiles(C_out / 16) * 16 + 16 + 32 * (b.steps[2] - 1 + ahead));
  if (C == b.variant) {  // constant taps: from the last of the tile's pixels that has a place
    const int pixel = odd(C / 16) * 16;
    int at = b.off_patch + (b.rows - 3) * b.row_pitch + (b.tw - 1) * pixel + 16;
    for (int row = 0; row < 3; ++row) {
      read(at + 2 * pixel + C - 32);
      read(at + row_below(row, b.row_pitch) + 32 * (ahead - 1));
      at += b.row_pitch;
    }
  }
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

}  // extern "C"
