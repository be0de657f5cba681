// Entropy (KL-divergence) calibration: _contrib_calibrate_entropy of the reference
// (src/operator/quantization/calibrate.cc:33-186), called by the histogram collector
// (python/mxnet/contrib/quantization.py:262-285).  All arithmetic is binary32 in the
// reference's order of operations, so the chosen threshold is the same number.
//
// The search is a serial chain of float additions per candidate threshold, 4000 candidates of
// up to 8001 bins each.  What bounds it is the logarithm of every non-empty bin of every
// candidate.  So:
//   - a candidate costs its non-empty bins, not its width.  Everything that is a sum of counts
//     (levels, non-empty bins of a level, the outliers folded into the edge bins) comes from
//     prefix sums, and a run of empty bins adds one constant to each of the three running
//     sums, which AddRepeated does in a few steps with the roundings that the single additions
//     make;
//   - candidates are independent: threads take them in blocks, from all the histograms of one
//     call.
// One histogram of 1.5 million values in 8001 bins: 155 ms in a straight restatement,
// 9 ms on 16 threads this way.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <limits>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "mxq_graph_pass.h"
#include "mxq_shim.h"

namespace mxq_graph {

namespace {

constexpr float kEps = 0.0001f;

uint32_t Bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, sizeof(u));
  return u;
}

// s + c + c + ... (n times), every addition rounded to nearest.  While the sum stays inside
// one binade its spacing is constant, so an addition moves it by the same amount each time
// (c rounded to that spacing) unless c lies exactly between two multiples of the spacing,
// where the direction depends on the sum's last bit.  Such ties, and the steps around a
// change of binade, are taken one by one.
float AddRepeated(float s, float c, size_t n) {
  while (n > 0) {
    const float t = s + c;
    --n;
    if (n < 4) {
      s = t;
      continue;
    }
    if (t == s) return s;
    const uint32_t bs = Bits(s) >> 23, bt = Bits(t) >> 23;  // sign and exponent
    const uint32_t exponent = bt & 0xffu;
    if (bs != bt || exponent < 64 || exponent > 250) {
      s = t;
      continue;
    }
    const double spacing = std::ldexp(1.0, static_cast<int>(exponent) - 150);
    const double step = static_cast<double>(t) - static_cast<double>(s);
    if (std::fabs(static_cast<double>(c) - step) >= 0.5 * spacing) {
      s = t;
      continue;
    }
    // steps that keep the magnitude inside [2^e, 2^(e+1)) with two steps to spare at the end
    const double low = std::ldexp(1.0, static_cast<int>(exponent) - 127);
    const double magnitude = std::fabs(static_cast<double>(t));
    const bool grows = (step > 0) == (t > 0);
    const double room = ((grows ? 2.0 * low - magnitude : magnitude - low) / std::fabs(step)) - 2.0;
    if (!(room >= 1.0)) {
      s = t;
      continue;
    }
    const size_t steps = room < static_cast<double>(n) ? static_cast<size_t>(room) : n;
    // multiples of the spacing below 2^24 of them: exact
    s = static_cast<float>(static_cast<double>(t) + static_cast<double>(steps) * step);
    n -= steps;
  }
  return s;
}

// One histogram and what all of its candidates read.
struct Problem {
  const float* hist;
  const float* edges;
  size_t bins;
  long zero_bin, half;  // candidate i in [half, zero_bin] keeps bins zero_bin - i .. zero_bin + i
  size_t levels;
  std::vector<float> head;        // head[j]: hist[0] + ... + hist[j], in that order
  std::vector<float> tail;        // tail[j]: hist[j] + ... + hist[bins - 1]; empty: not exact
  std::vector<long long> counts;  // counts[j]: sum of the integer parts of hist[0 .. j-1]
  std::vector<uint32_t> filled;   // filled[j]: bins below j whose integer part is not zero
  std::vector<uint32_t> seen;     // seen[j]: bins below j that are not zero
  std::vector<uint32_t> where;    // positions of the bins that are not zero
  std::vector<float> divergences;

  size_t candidates() const { return static_cast<size_t>(zero_bin + 1 - half); }

  Problem(const float* h, const float* e, size_t n, int num_quantized_bins)
      : hist(h), edges(e), bins(n) {
    CHECK(n % 2 == 1) << "the histogram needs an odd number of bins";
    CHECK(num_quantized_bins >= 1 && static_cast<size_t>(num_quantized_bins) <= n)
        << "num_quantized_bins out of range";
    zero_bin = static_cast<long>(n / 2);
    half = num_quantized_bins / 2;
    levels = static_cast<size_t>(num_quantized_bins);
    divergences.assign(candidates(), 0.f);
    head.resize(n);
    counts.assign(n + 1, 0);
    filled.assign(n + 1, 0);
    seen.assign(n + 1, 0);
    float sum = 0.f;
    bool whole = true;
    for (size_t j = 0; j < n; ++j) {
      head[j] = sum += h[j];
      const size_t count = static_cast<size_t>(h[j]);
      whole = whole && static_cast<float>(count) == h[j];
      counts[j + 1] = counts[j] + static_cast<long long>(count);
      filled[j + 1] = filled[j] + (count != 0);
      seen[j + 1] = seen[j] + (h[j] != 0.f);
      if (h[j] != 0.f) where.push_back(static_cast<uint32_t>(j));
    }
    // whole counts of less than 2^24 in all: every partial sum is exact in any order
    if (whole && counts[n] < (1LL << 24)) {
      tail.resize(n + 1);
      for (size_t j = 0; j <= n; ++j) tail[j] = static_cast<float>(counts[n] - counts[j]);
    }
  }
};

// Correction of a smoothed distribution: zeros become eps, the same mass comes off the other
// entries (calibrate.cc:33-64).  False: all entries are zero, or so many that it reaches 1.
bool Smoothing(size_t width, size_t nonzeros, float* take) {
  if (nonzeros == 0) return false;
  *take = kEps * static_cast<float>(width - nonzeros) / static_cast<float>(nonzeros);
  return !(*take >= 1.0);
}

// The non-zero entries of one candidate's reference distribution p, in order.
struct Scratch {
  std::vector<float> p, q;      // entry, and its value in the quantized distribution
  std::vector<uint32_t> empty;  // zero entries in front of it
  explicit Scratch(size_t n) : p(n + 2), q(n + 2), empty(n + 2) {}
};

// Divergence of candidate i; +inf where the quantized distribution cannot be smoothed.
float CandidateDivergence(const Problem& m, long i, Scratch* s) {
  const size_t start = static_cast<size_t>(m.zero_bin - i);
  const size_t stop = static_cast<size_t>(m.zero_bin + i + 1);
  const size_t width = stop - start;
  // everything outside is folded into the two edge entries of p
  float first = m.head[start], last = 0.f;
  if (width == 1) {
    for (size_t j = stop; j < m.bins; ++j) first += m.hist[j];
  } else if (!m.tail.empty()) {
    last = m.tail[stop - 1];
  } else {
    last = m.hist[stop - 1];
    for (size_t j = stop; j < m.bins; ++j) last += m.hist[j];
  }
  // q: the kept bins merged into `levels` levels (the last level takes the remainder), then
  // spread back evenly over the non-empty bins of each level.  The first edge entry counts
  // nothing there: its own bin belongs to the folded part.
  const size_t merged = width / m.levels;
  const size_t inner = start + 1;
  auto count_of = [&](size_t lo, size_t hi) {  // offsets from start
    lo += start;
    hi += start;
    if (lo < inner) lo = inner;
    return lo < hi ? m.counts[hi] - m.counts[lo] : 0LL;
  };
  auto filled_of = [&](size_t lo, size_t hi) {
    lo += start;
    hi += start;
    if (lo < inner) lo = inner;
    return lo < hi ? static_cast<int>(m.filled[hi] - m.filled[lo]) : 0;
  };
  size_t n = 0, q_nonzeros = 0;
  size_t before = 0;  // offset behind the last entry written
  auto put = [&](size_t offset, float p, float q) {
    s->empty[n] = static_cast<uint32_t>(offset - before);
    s->p[n] = p;
    s->q[n] = q;
    before = offset + 1;
    q_nonzeros += q != 0.f;
    ++n;
  };
  for (size_t j = 0; j < m.levels; ++j) {
    const size_t lo = j * merged;
    const bool final_level = j + 1 == m.levels;
    const size_t hi = final_level ? width : lo + merged;
    float level = static_cast<float>(static_cast<int>(count_of(lo, lo + merged)));
    if (final_level) level += static_cast<float>(static_cast<int>(count_of(lo + merged, width)));
    const int nonempty = filled_of(lo, hi);
    const float each = nonempty != 0 ? level / nonempty : 0.f;
    if (j == 0 && first != 0.f) put(0, first, each);
    // the bins strictly between the edge entries
    const size_t from = start + lo < inner ? inner : start + lo;
    const size_t to = start + hi > stop - 1 ? stop - 1 : start + hi;
    if (from < to)
      for (uint32_t k = m.seen[from]; k < m.seen[to]; ++k)
        put(m.where[k] - start, m.hist[m.where[k]], each);
    if (final_level && width > 1 && last != 0.f) put(width - 1, last, each);
  }
  const uint32_t empty_end = static_cast<uint32_t>(width - before);

  float p_take = 0.f, q_take = 0.f;
  if (!Smoothing(width, q_nonzeros, &q_take)) return std::numeric_limits<float>::infinity();
  CHECK(Smoothing(width, n, &p_take)) << "the reference distribution cannot be smoothed";
  float p_sum = 0.f, q_sum = 0.f;
  for (size_t k = 0; k < n; ++k) {
    if (s->empty[k] != 0) {
      p_sum = AddRepeated(p_sum, kEps, s->empty[k]);
      q_sum = AddRepeated(q_sum, kEps, s->empty[k]);
    }
    p_sum += s->p[k] -= p_take;
    s->q[k] = s->q[k] != 0.f ? s->q[k] - q_take : kEps;
    q_sum += s->q[k];
  }
  p_sum = AddRepeated(p_sum, kEps, empty_end);
  q_sum = AddRepeated(q_sum, kEps, empty_end);

  // KL(p || q) of the two after normalising each (calibrate.cc:66-87)
  float lowest = 1.f;
  for (size_t k = 0; k < n; ++k) {
    const float p = s->p[k] / p_sum, q = s->q[k] / q_sum;
    lowest = std::min(lowest, std::min(p, q));
    s->p[k] = p;
    s->q[k] = p / q;
  }
  CHECK(lowest > 0) << "p[i] > 0 && q[i] > 0";
  const float p_zero = kEps / p_sum, q_zero = kEps / q_sum;
  const float zero_term = p_zero * std::log(p_zero / q_zero);
  float kl = 0.f;
  for (size_t k = 0; k < n; ++k) {
    if (s->empty[k] != 0) kl = AddRepeated(kl, zero_term, s->empty[k]);
    kl += s->p[k] * std::log(s->q[k]);
  }
  return AddRepeated(kl, zero_term, empty_end);
}

// Threads a call may use: the CPUs this process may run on, OMP_NUM_THREADS where it is set,
// and no more than 16 (the search of one histogram is about 10 ms there).
unsigned ThreadLimit() {
  unsigned n = std::thread::hardware_concurrency();
  cpu_set_t set;
  CPU_ZERO(&set);
  if (sched_getaffinity(0, sizeof(set), &set) == 0) n = static_cast<unsigned>(CPU_COUNT(&set));
  if (const char* text = std::getenv("OMP_NUM_THREADS")) {
    const int asked = std::atoi(text);
    if (asked > 0 && static_cast<unsigned>(asked) < n) n = static_cast<unsigned>(asked);
  }
  return n < 1 ? 1 : n > 16 ? 16 : n;
}

}  // namespace

void CalibrateEntropyMany(size_t count, const float* const* hist, const float* const* hist_edges,
                          const size_t* num_bins, const int* num_quantized_bins,
                          float* thresholds, float* divergences) {
  std::vector<Problem> problems;
  problems.reserve(count);
  size_t widest = 0;
  for (size_t i = 0; i < count; ++i) {
    problems.emplace_back(hist[i], hist_edges[i], num_bins[i], num_quantized_bins[i]);
    widest = std::max(widest, num_bins[i]);
  }
  // blocks of candidates over all the problems, the widest candidates first
  constexpr size_t kBlock = 16;
  struct Block {
    Problem* problem;
    size_t first, end;  // candidate numbers, from the widest down
  };
  std::vector<Block> blocks;
  for (Problem& p : problems)
    for (size_t c = 0; c < p.candidates(); c += kBlock)
      blocks.push_back({&p, c, std::min(c + kBlock, p.candidates())});
  std::stable_sort(blocks.begin(), blocks.end(), [](const Block& a, const Block& b) {
    return a.problem->zero_bin - static_cast<long>(a.first) >
           b.problem->zero_bin - static_cast<long>(b.first);
  });
  std::atomic<size_t> next{0};
  std::mutex failure_lock;
  std::exception_ptr failure;
  auto work = [&]() {
    try {
      Scratch scratch(widest);
      for (size_t b = next++; b < blocks.size(); b = next++)
        for (size_t c = blocks[b].first; c < blocks[b].end; ++c) {
          Problem& p = *blocks[b].problem;
          const long i = p.zero_bin - static_cast<long>(c);
          p.divergences[i - p.half] = CandidateDivergence(p, i, &scratch);
        }
    } catch (...) {
      std::lock_guard<std::mutex> lock(failure_lock);
      if (!failure) failure = std::current_exception();
      next = blocks.size();
    }
  };
  std::vector<std::thread> threads;
  const size_t want = std::min<size_t>(ThreadLimit(), (blocks.size() + 3) / 4);
  for (size_t t = 1; t < want; ++t) {
    try {
      threads.emplace_back(work);
    } catch (const std::system_error&) {  // no more threads to be had: those that are there do
      break;
    }
  }
  work();
  for (std::thread& t : threads) t.join();
  if (failure) std::rethrow_exception(failure);

  for (size_t n = 0; n < count; ++n) {
    const Problem& p = problems[n];
    size_t best = 0;
    float best_divergence = std::numeric_limits<float>::max();
    for (size_t i = 0; i < p.divergences.size(); ++i) {
      if (p.divergences[i] < best_divergence) {
        best_divergence = p.divergences[i];
        best = i;
      }
    }
    divergences[n] = best_divergence;
    thresholds[n] = p.edges[p.zero_bin + p.half + static_cast<long>(best) + 1];
  }
}

void CalibrateEntropy(const float* hist, const float* hist_edges, size_t num_bins,
                      int num_quantized_bins, float* threshold, float* divergence) {
  CalibrateEntropyMany(1, &hist, &hist_edges, &num_bins, &num_quantized_bins, threshold,
                       divergence);
}

}  // namespace mxq_graph
