// Bounds of every candidate's divergence in the entropy calibration (_contrib_calibrate_entropy,
// src/operator/quantization/calibrate.cc:33-186), from which the host picks the few candidates it
// has to sum up in float itself (host/mxq_calibrate.cc, which defines a candidate, its levels, its
// two smoothed distributions and the order of the sums).
//
// What the divergence depends on in float are the two normalisations: chains of up to `bins`
// additions, taken here in the same order, a lane per candidate (thousands of chains side by side:
// what 16 host threads need 4 ms for).  The terms themselves are then summed up in double from the
// same float quotients, a wave per candidate, 256 bins at a time with their running sums: what the
// float chain can differ from that by is bounded by the roundings of its terms and of its additions,
// each one of the running sum it rounds.  Any bounds a few times wider cost the host a multiple of
// the candidates (its own, from sums of magnitudes only, leave 10 % of them).
//
// Three histograms of 8001 bins, 11622 candidates, with 16 host threads: 7.5 ms of search become 0.4
// of launches and 0.4 of sums on the host.  In all, ms, the host's own bounds / these: three of 2^25
// counts 5.5 / 1.2, one of 32767 bins 20 / 3.3, one of 8001 bins of which 20 are filled 1.5 / 1.0.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../../include/mxq.h"
#include "mxq_common.h"

namespace mxq {
namespace {

constexpr float kEps = 0.0001f;
constexpr int kMaxBins = 32767;     // a histogram in LDS
constexpr int kMaxProblems = 16;    // of one set of launches: their descriptions are an argument

struct Problem {
  int hist;       // where its bins begin
  int bins, levels, half, zero, candidates;
  int prefix;     // where its prefix sums begin
  int candidate;  // where its candidates begin
  long long level;  // where their levels begin
};
struct Info {     // of a candidate
  float first, last, p_take, q_take, p_sum, q_sum;
  float q_least;  // the least level that is not 0, smoothed
  int state;      // 0: bounded, 1: infinite, 2: unknown (the host's chain reports what is wrong)
};
struct Args {
  Problem p[kMaxProblems];
  const float* hist;
  int *counts, *filled, *seen;  // prefix sums of the integer parts, of them that are not 0, of bins
  float* head;                  // float sums from the first bin on
  int* exact;                   // per problem: every partial sum of counts is exact
  float* least;                 // ... the least bin that is not 0, 0 where one is below
  float* levels;                // [candidate][level], not smoothed
  Info* info;
  double* bounds;               // [candidate][2]
};

// s plus the values at `v` from `from` up to `to`, one after the other, with reads ahead of the
// additions; `each` is told every sum.  (A histogram of 2^24 counts and more, one of 8001 / 32767 bins:
// 0.08 / 0.34 ms of prefix sums and 0.08 / 0.96 of levels; a memory access at a time, 1.1 / 4.7 more.)
template <typename F>
__device__ __forceinline__ float chain(float s, const float* v, int from, int to, F each) {
  constexpr int B = 16;
  int j = from;
  for (; j + B <= to; j += B) {
    float x[B];
#pragma unroll
    for (int k = 0; k < B; ++k) x[k] = v[j + k];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      s += x[k];
      each(j + k, s);
    }
  }
  for (; j < to; ++j) {
    s += v[j];
    each(j, s);
  }
  return s;
}

// Prefix sums of one histogram, a contiguous run of bins per thread; the histogram in LDS, where
// the float sums of one that is not exact, which one thread adds up, replace it.
__global__ __launch_bounds__(1024) void entropy_prefix_kernel(Args a) {
  extern __shared__ float h[];
  const Problem p = a.p[blockIdx.x];
  const int tid = threadIdx.x, per = (p.bins + 1023) / 1024;
  const int from = tid * per < p.bins ? tid * per : p.bins;
  const int to = from + per < p.bins ? from + per : p.bins;
  __shared__ int sums[3][1024];
  for (int j = tid; j < p.bins; j += 1024) h[j] = a.hist[p.hist + j];
  __syncthreads();
  int s[3] = {0, 0, 0};
  bool whole = true;
  float least = INFINITY;
  for (int j = from; j < to; ++j) {
    const int n = static_cast<int>(h[j]);
    whole = whole && static_cast<float>(n) == h[j];
    if (h[j] != 0.0f) least = fminf(least, h[j]);
    s[0] += n;
    s[1] += n != 0;
    s[2] += h[j] != 0.0f;
  }
  for (int k = 0; k < 3; ++k) sums[k][tid] = s[k];
  whole = __syncthreads_and(whole) != 0;
  __shared__ float leasts[16];
  for (int d = 1; d < 64; d *= 2) least = fminf(least, __shfl_xor(least, d));
  if ((tid & 63) == 0) leasts[tid >> 6] = least;
  for (int step = 1; step < 1024; step *= 2) {
    int add[3];
    for (int k = 0; k < 3; ++k) add[k] = tid >= step ? sums[k][tid - step] : 0;
    __syncthreads();
    for (int k = 0; k < 3; ++k) sums[k][tid] += add[k];
    __syncthreads();
  }
  const int total = sums[0][1023];
  const bool exact = whole && total < (1 << 24);
  int at[3];
  for (int k = 0; k < 3; ++k) at[k] = sums[k][tid] - s[k];
  int* const out[3] = {a.counts + p.prefix, a.filled + p.prefix, a.seen + p.prefix};
  for (int j = from; j < to; ++j) {
    for (int k = 0; k < 3; ++k) out[k][j] = at[k];
    const int n = static_cast<int>(h[j]);
    at[0] += n;
    at[1] += n != 0;
    at[2] += h[j] != 0.0f;
    if (exact) a.head[p.prefix + j] = static_cast<float>(at[0]);
  }
  if (tid == 1023)
    for (int k = 0; k < 3; ++k) out[k][p.bins] = sums[k][1023];
  if (tid == 0) {
    a.exact[blockIdx.x] = exact;
    for (int k = 1; k < 16; ++k) least = fminf(least, leasts[k]);
    a.least[blockIdx.x] = fmaxf(least, 0.0f);
  }
  if (exact) return;
  __syncthreads();
  if (tid == 0) chain(0.0f, h, 0, p.bins, [&](int j, float sum) { h[j] = sum; });
  __syncthreads();
  for (int j = tid; j < p.bins; j += 1024) a.head[p.prefix + j] = h[j];
}

__device__ __forceinline__ int wave_sum(int v) {
  for (int d = 1; d < 64; d *= 2) v += __shfl_xor(v, d);
  return v;
}

// Correction of a smoothed distribution; false: all entries are zero, or so many that it reaches 1.
__device__ __forceinline__ bool smoothing(int width, int nonzeros, float* take) {
  if (nonzeros == 0) return false;
  *take = kEps * static_cast<float>(width - nonzeros) / static_cast<float>(nonzeros);
  return !(*take >= 1.0f);
}

// Levels, edge entries and smoothing of a candidate: a wave each, a level per lane.
__global__ __launch_bounds__(256) void entropy_levels_kernel(Args a) {
  const Problem p = a.p[blockIdx.y];
  const int lane = threadIdx.x & 63, s = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (s >= p.candidates) return;
  const int i = p.half + s, start = p.zero - i, stop = p.zero + i + 1;
  const int width = stop - start, merged = width / p.levels, inner = start + 1;
  const int* const counts = a.counts + p.prefix;
  const int* const filled = a.filled + p.prefix;
  const int* const seen = a.seen + p.prefix;
  const float first = a.head[p.prefix + start];
  float last;
  if (a.exact[blockIdx.y]) {
    last = static_cast<float>(counts[p.bins] - counts[stop - 1]);
  } else {
    const float* const h = a.hist + p.hist;
    last = chain(h[stop - 1], h, stop, p.bins, [](int, float) {});
  }
  auto between = [&](const int* sum, int lo, int hi) {
    return lo < hi ? sum[hi] - sum[lo] : 0;
  };
  int p_entries = 0, q_entries = 0;
  float least = INFINITY;
  float* const levels = a.levels + p.level + static_cast<long long>(s) * p.levels;
  for (int j = lane; j < p.levels; j += 64) {
    const int lo = j * merged, end = j + 1 == p.levels ? width : lo + merged;
    const int from = lo + start > inner ? lo + start : inner;
    float level = static_cast<float>(between(counts, from, lo + merged + start));
    if (j + 1 == p.levels) {
      const int rest = lo + merged + start > inner ? lo + merged + start : inner;
      level += static_cast<float>(between(counts, rest, stop));
    }
    const int nonempty = between(filled, from, end + start);
    level = nonempty != 0 ? level / static_cast<float>(nonempty) : 0.0f;
    levels[j] = level;
    const int to = end + start < stop - 1 ? end + start : stop - 1;
    const int entries = between(seen, from, to);
    p_entries += entries;
    if (level != 0.0f) {
      q_entries += entries + (j == 0 && first != 0.0f) + (j + 1 == p.levels && last != 0.0f);
      least = fminf(least, level);
    }
  }
  p_entries = wave_sum(p_entries) + (first != 0.0f) + (last != 0.0f);
  q_entries = wave_sum(q_entries);
  for (int d = 1; d < 64; d *= 2) least = fminf(least, __shfl_xor(least, d));
  if (lane == 0) {
    Info r = {};
    r.first = first;
    r.last = last;
    if (!smoothing(width, q_entries, &r.q_take))
      r.state = 1;
    else if (!smoothing(width, p_entries, &r.p_take))
      r.state = 2;
    r.q_least = least - r.q_take;
    a.info[p.candidate + s] = r;
  }
}

// The two float chains of a candidate, a lane each, of two waves; neighbouring candidates side by
// side.  A chain's pace is what its wave issues, an instruction every four clocks, and what it waits for,
// so a bin is an entry, one instruction that smooths it and the addition:
//   the distribution itself: every lane at the same bin, which a scalar load brings.  Smoothed it is
//     max(bin - take, kEps) where no bin but 0 is that small;
//   the levels: every lane at the same place of its own levels, which are as long as each other's or a
//     bin longer; in LDS a bin is infinity, or kEps where it is 0, and min(bin, level) is what it adds
//     where no level is below kEps.
// Where that does not hold a comparison and a selection smooth a bin, and each lane goes its own way
// through its levels.
// (For three histograms of 8001 bins: 165 us with both from LDS, smoothed by a comparison and a
// selection, and a level asked for one level ahead; 80 us so, and 122 for 135 where lanes go their own
// way, at 40 levels.)
typedef const __attribute__((address_space(4))) float* ScalarFloats;
constexpr int kMarksBehind = 64;  // what is read ahead past a lane's last bin

__device__ __forceinline__ float smoothed(float v, float take) {
  return v != 0.0f ? v - take : kEps;
}
// bins `from` ... `to` - 1 of the distribution, where the lane's own are from `mine` up to `last`
template <bool ALL, bool LARGE>
__device__ __forceinline__ void add_bins(float& sum, ScalarFloats h, int from, int to, int mine,
                                         int last, float take) {
  auto add = [&](int j, float v) {
    const float next = sum + (LARGE ? fmaxf(v - take, kEps) : smoothed(v, take));
    sum = ALL || (j >= mine && j < last) ? next : sum;
  };
  // two sets of bins take turns
  constexpr int B = 16;
  float x[B], y[B];
  auto read = [&](float (&v)[B], int j) {
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = h[j + k];
  };
  int j = from;
  if (j + 2 * B <= to) {
    read(x, j);
    for (; j + 2 * B <= to; j += 2 * B) {
      read(y, j + B);
#pragma unroll
      for (int k = 0; k < B; ++k) add(j + k, x[k]);
      if (j + 3 * B <= to) read(x, j + 2 * B);
#pragma unroll
      for (int k = 0; k < B; ++k) add(j + B + k, y[k]);
    }
  }
  for (; j < to; j += 8) {
    float z[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) z[k] = h[j + k < to ? j + k : to - 1];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (j + k < to) add(j + k, z[k]);
  }
}
template <bool LARGE>
__device__ __forceinline__ float p_chain(const Args& a, const Problem& p, const Info& r, int i) {
  const float take = r.p_take;
  float sum = smoothed(r.first, take);
  const int start = p.zero - i, stop = p.zero + i + 1;
  // the bins of lane 0, the widest, around those of the last lane, which are everyone's
  const int widest = __builtin_amdgcn_readfirstlane(i);
  const int narrowest = __builtin_amdgcn_readlane(i, 63);
  const int begin = p.zero - widest + 1, end = p.zero + widest;
  const int in = p.zero - narrowest + 1, out = p.zero + narrowest;
  const ScalarFloats h = reinterpret_cast<ScalarFloats>(
      reinterpret_cast<uintptr_t>(a.hist + p.hist));
  add_bins<false, LARGE>(sum, h, begin, in, start + 1, stop - 1, take);
  add_bins<true, LARGE>(sum, h, in, out, 0, 0, take);
  add_bins<false, LARGE>(sum, h, out, end, start + 1, stop - 1, take);
  return sum + smoothed(r.last, take);
}
// (positive floats are ordered as their bits are; fminf would have every mark made canonical first)
__device__ __forceinline__ float marked(int mark, float q) {
  const int level = __float_as_int(q);
  return __int_as_float(mark < level ? mark : level);
}
// Levels of 16 * k + REST bins (LONG: k > 0) in every lane, a bin longer where `more`.  A level's bins are
// added in a piece of REST, pieces of 16 and that bin, each read while what is before it is added.
template <int REST, bool LONG>
__device__ __forceinline__ float q_chain(const Problem& p, const Info& r, const float* levels,
                                         const int* marks, int width, int each, bool more) {
  const float take = r.q_take;
  const int step = each + static_cast<int>(more), full = each / 16;
  const int first = __float_as_int(r.first != 0.0f ? INFINITY : kEps);
  const int* v = marks;
  int x[16], y[16], last;
#pragma unroll
  for (int k = 0; k < REST; ++k) x[k] = k == 0 ? first : v[k];
#pragma unroll
  for (int k = 0; k < 16; ++k) y[k] = LONG ? (REST + k == 0 ? first : v[REST + k]) : 0;
  last = v[each];
  float sum = 0.0f;
  constexpr int B = 8;  // levels on their way
  float next[B];
#pragma unroll
  for (int k = 0; k < B; ++k) next[k] = levels[k < p.levels ? k : p.levels - 1];
  for (int j = 0; j < p.levels - 1; j += B) {
    float now[B];
#pragma unroll
    for (int k = 0; k < B; ++k) now[k] = smoothed(next[k], take);
#pragma unroll
    for (int k = 0; k < B; ++k)
      next[k] = levels[j + B + k < p.levels ? j + B + k : p.levels - 1];
    const int count = p.levels - 1 - j < B ? p.levels - 1 - j : B;
    for (int l = 0; l < count; ++l) {
      const float q = now[0];
#pragma unroll
      for (int k = 0; k + 1 < B; ++k) now[k] = now[k + 1];
#pragma unroll
      for (int k = 0; k < REST; ++k) sum += marked(x[k], q);
      __builtin_amdgcn_sched_barrier(0);
      const int* at = v + REST;
      v += step;
#pragma unroll
      for (int k = 0; k < REST; ++k) x[k] = v[k];
      if (LONG) {
        int left = full;
        do {
          at = --left > 0 ? at + 16 : v + REST;
#pragma unroll
          for (int half = 0; half < 16; half += 8) {
#pragma unroll
            for (int k = half; k < half + 8; ++k) sum += marked(y[k], q);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = half; k < half + 8; ++k) y[k] = at[k];
          }
        } while (left > 0);
      }
      sum = more ? sum + marked(last, q) : sum;
      last = v[each];
    }
  }
  // the last level is as long as it is
  const float q = smoothed(levels[p.levels - 1], take);
  const int mine = width - 1 - (p.levels - 1) * step;
  int longest = mine;
  for (int d = 1; d < 64; d *= 2) {
    const int other = __shfl_xor(longest, d);
    longest = other > longest ? other : longest;
  }
  longest = __builtin_amdgcn_readfirstlane(longest);
  for (int o = 0; o < longest; o += 16) {
#pragma unroll
    for (int k = 0; k < 16; ++k) y[k] = v[o + k < mine ? o + k : mine];
#pragma unroll
    for (int k = 0; k < 16; ++k) sum = o + k < mine ? sum + marked(y[k], q) : sum;
  }
  return sum + (r.last != 0.0f ? q : kEps);
}
template <int REST = 0>
__device__ __forceinline__ float q_chain_of(const Problem& p, const Info& r, const float* levels,
                                            const int* marks, int width, int each, bool more) {
  if constexpr (REST == 16) {
    return 0.0f;
  } else {
    if (each % 16 != REST)
      return q_chain_of<REST + 1>(p, r, levels, marks, width, each, more);
    return each < 16 ? q_chain<REST, false>(p, r, levels, marks, width, each, more)
                     : q_chain<REST, true>(p, r, levels, marks, width, each, more);
  }
}
__global__ __launch_bounds__(128) void entropy_chains_kernel(Args a) {
  extern __shared__ int marks[];
  const Problem p = a.p[blockIdx.y];
  if (static_cast<int>(blockIdx.x) * 64 >= p.candidates) return;
  for (int j = threadIdx.x; j < p.bins; j += 128 * 16) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
      v[k] = a.hist[p.hist + (j + 128 * k < p.bins ? j + 128 * k : p.bins - 1)];
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (j + 128 * k < p.bins)
        marks[j + 128 * k] = __float_as_int(v[k] != 0.0f ? INFINITY : kEps);
  }
  __syncthreads();
  // the widest first: a wave of them takes longest; lanes without a candidate take the narrowest
  const int at = p.candidates - 1 - (blockIdx.x * 64 + (threadIdx.x & 63));
  const int s = at < 0 ? 0 : at;
  Info* const info = a.info + p.candidate + s;
  const Info r = *info;
  if (__all(r.state != 0)) return;
  const int i = p.half + s, width = 2 * i + 1;
  if (threadIdx.x < 64) {
    const float sum = __all(r.state != 0 || a.least[blockIdx.y] - r.p_take >= kEps)
                          ? p_chain<true>(a, p, r, i)
                          : p_chain<false>(a, p, r, i);
    if (r.state == 0 && at >= 0) info->p_sum = sum;
    return;
  }
  const float* const levels = a.levels + p.level + static_cast<long long>(s) * p.levels;
  const int merged = width / p.levels, each = __builtin_amdgcn_readlane(merged, 63);
  const int most = __builtin_amdgcn_readfirstlane(merged);
  const int* const mine = marks + p.zero - i;
  float sum;
  if (most <= each + 1 && __all(r.state != 0 || r.q_least >= kEps)) {
    sum = q_chain_of(p, r, levels, mine, width, each, merged > each);
  } else {
    float level = levels[0], q = smoothed(level, r.q_take);
    sum = r.first != 0.0f ? q : kEps;
    for (int j = 0; j < p.levels; ++j) {
      q = smoothed(level, r.q_take);
      const bool end = j + 1 == p.levels;
      if (!end) level = levels[j + 1];
      const int to = end ? width - 1 : (j + 1) * merged;
      int o = j == 0 ? 1 : j * merged;
      for (; o + 8 <= to; o += 8) {
        int v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = mine[o + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += v[k] == __float_as_int(kEps) ? kEps : q;
      }
      if (o < to) {  // fewer than 8, read in one go as well
        int v[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) v[k] = mine[o + k < to ? o + k : o];
#pragma unroll
        for (int k = 0; k < 7; ++k)
          if (o + k < to) sum += v[k] == __float_as_int(kEps) ? kEps : q;
      }
    }
    sum += r.last != 0.0f ? q : kEps;
  }
  if (r.state == 0 && at >= 0) info->q_sum = sum;
}

// a / b from a reciprocal, the first guess and one correction by its remainder (Markstein's division).
// With RN(1 / b) it is RN(a / b) while nothing leaves the normal range: in units of the quotient's last
// place u the guess is off by less than 1.5, so the remainder is rounded by no more than 1 / b of u 2^-23 and
// the correction misses a / b by less than 3.5 u 2^-24, while a quotient that is no midpoint of two floats is
// u 2^-24 n / b from the next one for a whole n.  That leaves those with n of up to 7, and a test goes
// through all of them.  With a reciprocal a last place off it is that, or where a / b is as close to a midpoint,
// the float on its other side.
__device__ __forceinline__ float quotient(float a, float b, float reciprocal) {
  const float q = a * reciprocal;
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), reciprocal, q);
}
// The natural logarithm of a normal positive number: the instruction's, a last place of log2, times
// ln 2 in two parts.
__device__ __forceinline__ float natural_log(float x) {
  constexpr float hi = 0x1.62e42ep-1f, lo = 0x1.efa39ep-25f;
  const float y = __builtin_amdgcn_logf(x), z = y * hi;
  return z + __builtin_fmaf(y, lo, __builtin_fmaf(y, hi, -z));
}

// The bounds, a wave per candidate, 16 bins in a row per lane.  With u = 2^-24, a term of the float
// chain carries a logarithm of at most a last place (2u) and a product's rounding, a term here a
// logarithm of at most two (4u; a test measures it on every normal number) and an exact product; a sum
// of the chain carries u of itself.  The factors are the chain's, and add up to one; the logarithms'
// arguments are its own or the next float, 2u of the logarithm.
// (Vector instructions bound it: 136 us for the three histograms above with the compiler's divisions and
// logarithm and 4 bins in a row, a scan of the wave for every 256 bins; 95 us so.)
__global__ __launch_bounds__(256) void entropy_bounds_kernel(Args a) {
  constexpr int B = 16;
  const Problem p = a.p[blockIdx.y];
  const int lane = threadIdx.x & 63, s = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (s >= p.candidates) return;
  double* const out = a.bounds + 2 * static_cast<long long>(p.candidate + s);
  const Info r = a.info[p.candidate + s];
  if (r.state != 0) {
    if (lane < 2) out[lane] = r.state == 1 || lane == 1 ? INFINITY : -INFINITY;
    return;
  }
  const int i = p.half + s, start = p.zero - i, width = 2 * i + 1, merged = width / p.levels;
  const float* const h = a.hist + p.hist + start;
  const float* const levels = a.levels + p.level + static_cast<long long>(s) * p.levels;
  const float p_once = 1.0f / r.p_sum, q_once = 1.0f / r.q_sum;
  const float p_zero = kEps / r.p_sum, q_zero = kEps / r.q_sum;
  const double zero_term = static_cast<double>(p_zero) * static_cast<double>(logf(p_zero / q_zero));
  double sum = 0.0;  // the same in every lane
  double magnitude = 0.0, sums = 0.0;
  bool bad = false;
  for (int base = 0; base < width; base += 64 * B) {
    const int from = base + B * lane;
    int j = from / merged, rest = from - j * merged;
    float v[B];
    double t[B];
    if (from + B <= width) {
#pragma unroll
      for (int k = 0; k < B; k += 4) __builtin_memcpy(v + k, h + from + k, 16);
    } else {
#pragma unroll
      for (int k = 0; k < B; ++k) v[k] = from + k < width ? h[from + k] : 0.0f;
    }
    double all = 0.0;
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const int o = from + k;
      const float x = o == 0 ? r.first : o + 1 == width ? r.last : v[k];
      const float level = levels[j < p.levels ? j : p.levels - 1];
      const float q = level != 0.0f ? level - r.q_take : kEps;
      const float pn = quotient(x - r.p_take, r.p_sum, p_once), qn = quotient(q, r.q_sum, q_once);
      const float once = __builtin_amdgcn_rcpf(qn);
      const double term =
          static_cast<double>(pn) * static_cast<double>(natural_log(quotient(pn, qn, once)));
      const bool filled = x != 0.0f && o < width;
      bad = bad || (filled && (!(pn > 0.0f) || !(qn > 0.0f)));
      t[k] = filled ? term : o < width ? zero_term : 0.0;
      magnitude += fabs(t[k]);
      all += t[k];
      if (++rest == merged) {
        ++j;
        rest = 0;
      }
    }
    double before = all;
    for (int d = 1; d < 64; d *= 2) {
      const double other = __shfl_up(before, d);
      before += lane >= d ? other : 0.0;
    }
    before += sum;
    sum = __shfl(before, 63);
    before -= all;
#pragma unroll
    for (int k = 0; k < B; ++k) {
      before += t[k];
      sums += from + k < width ? fabs(before) : 0.0;
    }
  }
  for (int d = 1; d < 64; d *= 2) {
    magnitude += __shfl_xor(magnitude, d);
    sums += __shfl_xor(sums, d);
  }
  bad = __any(bad);
  const double u = 1.0 / 16777216.0;
  // (5 % for what is of second order, the factors' sum among it)
  const double margin = 1.05 * u * (8.0 * magnitude + 2.0 + sums) + 1e-12;
  if (lane == 0) {
    const bool known = !bad && isfinite(sum) && isfinite(margin);
    out[0] = known ? sum - margin : -INFINITY;
    out[1] = known ? sum + margin : INFINITY;
  }
}

#ifdef MXQ_TEST_HOOKS
__global__ __launch_bounds__(256) void entropy_functions_kernel(const float* a, const float* b,
                                                                size_t n, float* exact, float* near,
                                                                float* logs) {
  const size_t i = blockIdx.x * size_t(256) + threadIdx.x;
  if (i >= n) return;
  if (exact != nullptr) exact[i] = quotient(a[i], b[i], 1.0f / b[i]);
  if (near != nullptr) near[i] = quotient(a[i], b[i], __builtin_amdgcn_rcpf(b[i]));
  if (logs != nullptr) logs[i] = natural_log(a[i]);
}
#endif

size_t up256(size_t x) { return (x + 255) / 256 * 256; }

// Where the parts of the workspace lie, and the problems' descriptions.
struct Layout {
  size_t prefix = 0, candidates = 0, levels = 0, hist = 0;  // elements
  size_t bytes = 0, at[8];
  Layout(int count, const int* bins, const int* num_levels, Problem* out) {
    for (int i = 0; i < count; ++i) {
      MXQ_CHECK(bins[i] % 2 == 1 && bins[i] <= kMaxBins && num_levels[i] >= 3 &&
                    num_levels[i] <= bins[i],
                "bins or levels out of range");
      Problem p;
      p.bins = bins[i];
      p.levels = num_levels[i];
      p.half = num_levels[i] / 2;
      p.zero = bins[i] / 2;
      p.candidates = p.zero + 1 - p.half;
      p.hist = static_cast<int>(hist);
      p.prefix = static_cast<int>(prefix);
      p.candidate = static_cast<int>(candidates);
      p.level = static_cast<long long>(levels);
      hist += bins[i];
      prefix += bins[i] + 1;
      candidates += p.candidates;
      levels += static_cast<size_t>(p.candidates) * p.levels;
      if (out != nullptr) out[i] = p;
    }
    const size_t parts[8] = {prefix * 4, prefix * 4, prefix * 4, prefix * 4, kMaxProblems * 4,
                             levels * 4, candidates * sizeof(Info), kMaxProblems * 4};
    for (int k = 0; k < 8; ++k) {
      at[k] = bytes;
      bytes += up256(parts[k]);
    }
  }
};

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" {

size_t mxq_entropy_bounds_workspace(int count, const int* bins, const int* levels) {
  try {
    if (count <= 0 || count > kMaxProblems || bins == nullptr || levels == nullptr) return 0;
    return Layout(count, bins, levels, nullptr).bytes;
  } catch (const std::exception& e) {
    set_last_error(e.what());
    return 0;
  }
}

int mxq_entropy_bounds(void* stream, int count, const float* hist, const int* bins,
                       const int* levels, double* bounds, void* workspace,
                       size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(count >= 0 && count <= kMaxProblems, "too many histograms");
  if (count == 0) return 0;
  MXQ_CHECK(hist && bins && levels && bounds && workspace, "null pointer");
  Args a;
  const Layout l(count, bins, levels, a.p);
  MXQ_CHECK(workspace_bytes >= l.bytes && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0,
            "workspace too small or unaligned");
  char* const ws = static_cast<char*>(workspace);
  a.hist = hist;
  a.counts = reinterpret_cast<int*>(ws + l.at[0]);
  a.filled = reinterpret_cast<int*>(ws + l.at[1]);
  a.seen = reinterpret_cast<int*>(ws + l.at[2]);
  a.head = reinterpret_cast<float*>(ws + l.at[3]);
  a.exact = reinterpret_cast<int*>(ws + l.at[4]);
  a.levels = reinterpret_cast<float*>(ws + l.at[5]);
  a.info = reinterpret_cast<Info*>(ws + l.at[6]);
  a.least = reinterpret_cast<float*>(ws + l.at[7]);
  a.bounds = bounds;
  int most = 0, widest = 0;
  for (int i = 0; i < count; ++i) {
    most = a.p[i].candidates > most ? a.p[i].candidates : most;
    widest = bins[i] > widest ? bins[i] : widest;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned n = static_cast<unsigned>(count);
  hipLaunchKernelGGL(entropy_prefix_kernel, dim3(n), dim3(1024), static_cast<size_t>(widest) * 4, s,
                     a);
  MXQ_LAUNCH_CHECK();
  hipLaunchKernelGGL(entropy_levels_kernel, dim3((most + 3) / 4, n), dim3(256), 0, s, a);
  MXQ_LAUNCH_CHECK();
  hipLaunchKernelGGL(entropy_chains_kernel, dim3((most + 63) / 64, n), dim3(128),
                     static_cast<size_t>(widest + kMarksBehind) * 4, s, a);
  MXQ_LAUNCH_CHECK();
  hipLaunchKernelGGL(entropy_bounds_kernel, dim3((most + 3) / 4, n), dim3(256), 0, s, a);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}

#ifdef MXQ_TEST_HOOKS
// tests/mxq_test_hooks.h
int mxq_test_entropy_functions(void* stream, const float* a, const float* b, size_t n, float* exact,
                               float* near, float* logs) {
  MXQ_API_BEGIN();
  if (n == 0) return 0;
  MXQ_CHECK(n <= (size_t(1) << 31), "too many numbers");
  MXQ_CHECK(a != nullptr && (b != nullptr || (exact == nullptr && near == nullptr)), "null pointer");
  hipLaunchKernelGGL(entropy_functions_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256),
                     0, static_cast<hipStream_t>(stream), a, b, n, exact, near, logs);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}
#endif  // MXQ_TEST_HOOKS

}  // extern "C"
