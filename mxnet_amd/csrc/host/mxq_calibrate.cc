// Entropy (KL-divergence) calibration: _contrib_calibrate_entropy of the reference
// (src/operator/quantization/calibrate.cc:33-186), called by the histogram collector
// (python/mxnet/contrib/quantization.py:262-285).  All arithmetic is binary32 in the
// reference's order of operations, so the chosen threshold is the same number.
//
// The search is a serial chain of float additions per candidate threshold, 4000 candidates of
// up to 8001 bins each, with a logarithm per non-empty bin.  So:
//   - everything that is a sum of counts (levels, non-empty bins of a level, the outliers folded
//     into the edge bins) comes from prefix sums;
//   - a candidate's divergence is first estimated in double precision from its two
//     normalisations (float chains, taken as they are) and prefix sums of h log h and its
//     derivatives: one logarithm per quantized level instead of one per bin.  A bound on what
//     the float chain can differ from that (Candidate::margin) leaves the few candidates that
//     can be the smallest, and only those are summed up in float.  Where a GPU is in use the
//     bounds come from there (csrc/mxq_entropy.hip), tighter ones: of 11622 candidates 1155 are
//     left by the estimate, and 3 (the smallest of each histogram) by those;
//   - a run of empty bins adds one constant to each of the running sums, which AddRepeated does
//     in a few steps with the roundings that the single additions make;
//   - candidates are independent: threads take them in blocks, from all the histograms of one
//     call.
// One histogram of 1.5 million values in 8001 bins on 16 threads: 155 ms in a straight
// restatement on one, 4.3 ms without the estimate, 2 ms this way.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <functional>
#include <limits>
#include <memory>
#include <mutex>
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

double PowerOfTwo(int e) {
  const uint64_t u = static_cast<uint64_t>(e + 1023) << 52;
  double d;
  std::memcpy(&d, &u, sizeof(d));
  return d;
}

constexpr size_t kRepeats = 14;

// s + c + c + ... (n times), every addition rounded to nearest.  While the sum stays inside
// one binade its spacing is constant, so an addition moves it by the same amount each time
// (c rounded to that spacing) unless c lies exactly between two multiples of the spacing,
// where the direction depends on the sum's last bit.  Such ties, and the steps around a
// change of binade, are taken one by one.
float AddRepeated(float s, float c, size_t n) {
  while (n > 0) {
    const float t = s + c;
    --n;
    if (n < kRepeats) {  // below what the steps underneath cost
      s = t;
      for (; n > 0; --n) s += c;
      return s;
    }
    if (t == s) return s;
    const uint32_t bs = Bits(s) >> 23, bt = Bits(t) >> 23;  // sign and exponent
    const uint32_t exponent = bt & 0xffu;
    if (bs != bt || exponent < 64 || exponent > 250) {
      s = t;
      continue;
    }
    const double low = PowerOfTwo(static_cast<int>(exponent) - 127);
    const double spacing = low * (1.0 / 8388608.0);
    const double step = static_cast<double>(t) - static_cast<double>(s);
    if (std::fabs(static_cast<double>(c) - step) >= 0.5 * spacing) {
      s = t;
      continue;
    }
    // steps that keep the magnitude inside [2^e, 2^(e+1)) with two steps to spare at the end
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
  std::vector<uint32_t> filled_run;  // bins that are not zero from where[k] on, without a gap
  std::vector<double> hlogh, logh, inv1, inv2, sum;  // over the first k entries of where
  bool estimable;                 // every bin that is not zero holds at least 1
  std::vector<double> lower, upper;  // bounds of the candidates' divergences
  std::vector<float> divergences;

  size_t candidates() const { return static_cast<size_t>(zero_bin + 1 - half); }

  Problem(const float* h, const float* e, size_t n, int num_quantized_bins, bool estimate)
      : hist(h), edges(e), bins(n) {
    CHECK(n % 2 == 1) << "the histogram needs an odd number of bins";
    CHECK(num_quantized_bins >= 1 && static_cast<size_t>(num_quantized_bins) <= n)
        << "num_quantized_bins out of range";
    zero_bin = static_cast<long>(n / 2);
    half = num_quantized_bins / 2;
    levels = static_cast<size_t>(num_quantized_bins);
    divergences.assign(candidates(), std::numeric_limits<float>::infinity());
    lower.assign(candidates(), std::numeric_limits<double>::infinity());
    upper = lower;
    head.resize(n);
    counts.assign(n + 1, 0);
    filled.assign(n + 1, 0);
    seen.assign(n + 1, 0);
    float running = 0.f;
    bool whole = true;
    for (size_t j = 0; j < n; ++j) {
      head[j] = running += h[j];
      const size_t count = static_cast<size_t>(h[j]);
      whole = whole && static_cast<float>(count) == h[j];
      counts[j + 1] = counts[j] + static_cast<long long>(count);
      filled[j + 1] = filled[j] + (count != 0);
      seen[j + 1] = seen[j] + (h[j] != 0.f);
      if (h[j] != 0.f) where.push_back(static_cast<uint32_t>(j));
    }
    filled_run.assign(where.size(), 1);
    for (size_t k = where.size(); k-- > 1;)
      if (where[k] == where[k - 1] + 1) filled_run[k - 1] = filled_run[k] + 1;
    estimable = estimate;
    if (estimate) Terms();
    // whole counts of less than 2^24 in all: every partial sum is exact in any order
    if (whole && counts[n] < (1LL << 24)) {
      tail.resize(n + 1);
      for (size_t j = 0; j <= n; ++j) tail[j] = static_cast<float>(counts[n] - counts[j]);
    }
  }

 private:
  void Terms() {
    for (std::vector<double>* v : {&hlogh, &logh, &inv1, &inv2, &sum}) {
      v->reserve(where.size() + 1);
      v->push_back(0.0);
    }
    for (const uint32_t j : where) {
      const double h0 = hist[j], l = std::log(h0);
      estimable = estimable && h0 >= 1.0 && std::isfinite(h0);
      hlogh.push_back(hlogh.back() + h0 * l);
      logh.push_back(logh.back() + l);
      inv1.push_back(inv1.back() + 1.0 / h0);
      inv2.push_back(inv2.back() + 1.0 / (h0 * h0));
      sum.push_back(sum.back() + h0);
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
  std::vector<float> p, q;      // entry, and its ratio to the quantized distribution
  std::vector<uint32_t> empty;  // zero entries in front of it
  std::vector<float> levels;
  explicit Scratch(size_t n) : p(n + 2), q(n + 2), empty(n + 2), levels(8 * n) {}
};

// What both evaluations of candidate i start from.
struct Candidate {
  size_t start, stop, width, merged, inner;
  float first, last;  // the edge entries of p: everything outside is folded into them

  Candidate(const Problem& m, long i) {
    start = static_cast<size_t>(m.zero_bin - i);
    stop = static_cast<size_t>(m.zero_bin + i + 1);
    width = stop - start;
    merged = width / m.levels;
    inner = start + 1;
    first = m.head[start];
    last = 0.f;
    if (width == 1) {
      for (size_t j = stop; j < m.bins; ++j) first += m.hist[j];
    } else if (!m.tail.empty()) {
      last = m.tail[stop - 1];
    } else {
      last = m.hist[stop - 1];
      for (size_t j = stop; j < m.bins; ++j) last += m.hist[j];
    }
  }
  // q: the kept bins merged into levels (the last level takes the remainder), then spread back
  // evenly over the non-empty bins of each level.  The first edge entry counts nothing there:
  // its own bin belongs to the folded part.  Offsets are from start.
  long long Counts(const Problem& m, size_t lo, size_t hi) const {
    lo = std::max(lo + start, inner);
    hi += start;
    return lo < hi ? m.counts[hi] - m.counts[lo] : 0LL;
  }
  int Filled(const Problem& m, size_t lo, size_t hi) const {
    lo = std::max(lo + start, inner);
    hi += start;
    return lo < hi ? static_cast<int>(m.filled[hi] - m.filled[lo]) : 0;
  }
  size_t LevelEnd(const Problem& m, size_t j) const {
    return j + 1 == m.levels ? width : (j + 1) * merged;
  }
  // the value of level j's non-empty bins
  float Level(const Problem& m, size_t j) const {
    const size_t lo = j * merged;
    float level = static_cast<float>(static_cast<int>(Counts(m, lo, lo + merged)));
    if (j + 1 == m.levels)
      level += static_cast<float>(static_cast<int>(Counts(m, lo + merged, width)));
    const int nonempty = Filled(m, lo, LevelEnd(m, j));
    return nonempty != 0 ? level / nonempty : 0.f;
  }
  // entries of where[] strictly between the edge entries that level j holds
  void Entries(const Problem& m, size_t j, uint32_t* k0, uint32_t* k1) const {
    const size_t from = std::max(start + j * merged, inner);
    const size_t to = std::min(start + LevelEnd(m, j), stop - 1);
    *k0 = from < to ? m.seen[from] : 0;
    *k1 = from < to ? m.seen[to] : 0;
  }
};

// The candidate's normalisations and what they are made of.
struct Sums {
  size_t p_entries, q_entries;  // non-zero ones
  float p_take, q_take, p_sum, q_sum;
};

// False: the quantized distribution cannot be smoothed (an infinite divergence).  levels[j] is
// the value of level j, then its smoothed value.
bool Normalise(const Problem& m, const Candidate& c, Sums* s, float* levels) {
  s->p_entries = c.first != 0.f;
  s->p_entries += c.width > 1 && c.last != 0.f;
  s->q_entries = 0;
  for (size_t j = 0; j < m.levels; ++j) {
    levels[j] = c.Level(m, j);
    uint32_t k0, k1;
    c.Entries(m, j, &k0, &k1);
    s->p_entries += k1 - k0;
    if (levels[j] != 0.f)
      s->q_entries += (k1 - k0) + (j == 0 && c.first != 0.f) +
                      (j + 1 == m.levels && c.width > 1 && c.last != 0.f);
  }
  if (!Smoothing(c.width, s->q_entries, &s->q_take)) return false;
  CHECK(Smoothing(c.width, s->p_entries, &s->p_take))
      << "the reference distribution cannot be smoothed";
  // the float sum of the smoothed quantized distribution; p's is PSums's
  float q_sum = 0.f;
  size_t before = 0;  // offset behind the last entry
  auto gap = [&](size_t offset) {
    q_sum = AddRepeated(q_sum, kEps, offset - before);
    before = offset + 1;
  };
  for (size_t j = 0; j < m.levels; ++j) {
    const float q = levels[j] = levels[j] != 0.f ? levels[j] - s->q_take : kEps;
    if (j == 0 && c.first != 0.f) {
      gap(0);
      q_sum += q;
    }
    uint32_t k0, k1;
    c.Entries(m, j, &k0, &k1);
    if (k0 < k1 && m.where[k1 - 1] - m.where[k0] == k1 - 1 - k0) {  // no empty bin among them
      gap(m.where[k0] - c.start);
      q_sum = AddRepeated(q_sum, q, k1 - k0);
      before = m.where[k1 - 1] - c.start + 1;
    } else {
      for (uint32_t k = k0; k < k1; ++k) {
        gap(m.where[k] - c.start);
        q_sum += q;
      }
    }
    if (j + 1 == m.levels && c.width > 1 && c.last != 0.f) {
      gap(c.width - 1);
      q_sum += q;
    }
  }
  gap(c.width);
  s->q_sum = q_sum;
  return true;
}

// The float sums of the smoothed reference distributions of `count` candidates, each one bin narrower
// on both sides than the one before: eight chains of additions side by side, which share the bins all of them keep.
constexpr int kLanes = 8;
typedef float Lanes __attribute__((vector_size(4 * kLanes)));

void PSums(const Problem& m, int count, const Candidate* c, const float* take,
           float* p_sum) {
  auto value = [&](int l, size_t at) {
    return at == c[l].start ? c[l].first : at + 1 == c[l].stop ? c[l].last : m.hist[at];
  };
  auto scalar = [&](int l, float sum, size_t from, size_t to) {
    for (size_t at = from; at < to; ++at) {
      const float v = value(l, at);
      sum += v != 0.f ? v - take[l] : kEps;
    }
    return sum;
  };
  // the bins strictly inside the narrowest of them
  const Candidate& narrow = c[count - 1];
  const size_t from = narrow.inner, to = narrow.stop - 1;
  if (narrow.width < 3) {
    for (int l = 0; l < count; ++l) p_sum[l] = scalar(l, 0.f, c[l].start, c[l].stop);
    return;
  }
  Lanes sum = {}, less = {};
  for (int l = 0; l < count; ++l) {
    sum[l] = scalar(l, 0.f, c[l].start, from);
    less[l] = take[l];
  }
  size_t before = from;
  auto gap = [&](size_t at) {
    const size_t n = at - before;
    before = at + 1;
    if (n < kRepeats) {
      for (size_t k = 0; k < n; ++k) sum += kEps;
    } else {
      for (int l = 0; l < count; ++l) sum[l] = AddRepeated(sum[l], kEps, n);
    }
  };
  for (uint32_t k = m.seen[from]; k < m.seen[to];) {
    gap(m.where[k]);
    // bins up to the next empty one
    const uint32_t end = std::min(m.seen[to], k + m.filled_run[k]);
    const float* h = m.hist + m.where[k];
    before = m.where[k] + (end - k);
    Lanes running = sum;
    for (; k < end; ++k) running += *h++ - less;
    sum = running;
  }
  gap(to);
  for (int l = 0; l < count; ++l) p_sum[l] = scalar(l, sum[l], to, c[l].stop);
}

// p[k] -> p[k] / p_sum, q[k] -> that over q[k] / q_sum; whether all four are positive.
__attribute__((optimize("O3"))) bool Ratios(float* __restrict__ p, float* __restrict__ q,
                                            size_t n, float p_sum, float q_sum) {
  int bad = 0;
  for (size_t k = 0; k < n; ++k) {
    const float a = p[k] / p_sum, b = q[k] / q_sum;
    bad |= static_cast<int>(!(a > 0)) | static_cast<int>(!(b > 0));
    p[k] = a;
    q[k] = a / b;
  }
  return bad == 0;
}

// The candidate's divergence as the float chain gives it (calibrate.cc:66-87).
float Divergence(const Problem& m, const Candidate& c, const Sums& s, const float* levels,
                 Scratch* scratch) {
  size_t n = 0, before = 0;
  auto put = [&](size_t offset, float entry, float level) {
    scratch->empty[n] = static_cast<uint32_t>(offset - before);
    before = offset + 1;
    scratch->p[n] = entry - s.p_take;
    scratch->q[n] = level;
    ++n;
  };
  for (size_t j = 0; j < m.levels; ++j) {
    if (j == 0 && c.first != 0.f) put(0, c.first, levels[j]);
    uint32_t k0, k1;
    c.Entries(m, j, &k0, &k1);
    for (uint32_t k = k0; k < k1; ++k) put(m.where[k] - c.start, m.hist[m.where[k]], levels[j]);
    if (j + 1 == m.levels && c.width > 1 && c.last != 0.f) put(c.width - 1, c.last, levels[j]);
  }
  CHECK(Ratios(scratch->p.data(), scratch->q.data(), n, s.p_sum, s.q_sum))
      << "p[i] > 0 && q[i] > 0";
  const float p_zero = kEps / s.p_sum, q_zero = kEps / s.q_sum;
  const float zero_term = p_zero * std::log(p_zero / q_zero);
  for (size_t k = 0; k < n; ++k) scratch->p[k] *= std::log(scratch->q[k]);
  float kl = 0.f;
  for (size_t k = 0; k < n; ++k) {
    if (scratch->empty[k] != 0) kl = AddRepeated(kl, zero_term, scratch->empty[k]);
    kl += scratch->p[k];
  }
  return AddRepeated(kl, zero_term, c.width - before);
}

// Bounds of what Divergence returns; (-inf, +inf) where none are known.
//
// With ps = h - take (eps for an empty bin), P its float sum, qs and Q likewise, the chain's
// exact counterpart is (sum ps log ps - sum ps log qs) / P + (sum ps / P) log(Q / P).  The second
// sum has one logarithm per level; the first is expanded in `take`, at most 0.01 against h >= 1:
// the terms past the third order are below 1e-9 of P.
//
// The chain's terms carry a few roundings each (u = 2^-24: 10u over all of them, and 6u of their
// magnitude), its additions one rounding of the running sum each, which never exceeds the sum S
// of the terms' magnitudes.  S = kl + 2 N with N the negative part, and N <= sum max(0, q - p),
// which Pinsker's inequality bounds by the divergence itself once p and q are scaled to sum to 1
// (a and b are their sums).
void Estimate(const Problem& m, const Candidate& c, const Sums& s, const float* levels,
              double* lower, double* upper) {
  *lower = -std::numeric_limits<double>::infinity();
  *upper = std::numeric_limits<double>::infinity();
  if (!m.estimable || s.p_take > 0.01f || c.width < 3) return;
  const double take = s.p_take, P = s.p_sum, Q = s.q_sum;
  double plogp = 0, plogq = 0, p_total = 0, q_total = 0;
  auto edge = [&](float entry) {
    if (entry == 0.f) return 0.0;
    const double p = static_cast<double>(entry) - take;
    plogp += p * std::log(p);
    p_total += p;
    return p;
  };
  const uint32_t k0 = m.seen[c.inner], k1 = m.seen[c.stop - 1];
  const double count = k1 - k0;
  plogp = (m.hlogh[k1] - m.hlogh[k0]) - take * (m.logh[k1] - m.logh[k0] + count) +
          take * take / 2 * (m.inv1[k1] - m.inv1[k0]) +
          take * take * take / 6 * (m.inv2[k1] - m.inv2[k0]);
  p_total = (m.sum[k1] - m.sum[k0]) - take * count;
  const double at_first = edge(c.first), at_last = edge(c.last);
  for (size_t j = 0; j < m.levels; ++j) {
    uint32_t e0, e1;
    c.Entries(m, j, &e0, &e1);
    double mass = (m.sum[e1] - m.sum[e0]) - take * static_cast<double>(e1 - e0);
    double entries = e1 - e0;
    if (j == 0 && c.first != 0.f) {
      mass += at_first;
      ++entries;
    }
    if (j + 1 == m.levels && c.last != 0.f) {
      mass += at_last;
      ++entries;
    }
    if (entries == 0) continue;
    const double q = levels[j];
    if (!(q > 0)) return;  // the chain reports it
    plogq += mass * std::log(q);
    q_total += entries * q;
  }
  const double empty = static_cast<double>(c.width - s.p_entries);
  p_total += empty * kEps;
  q_total += empty * kEps;
  if (!(P > 0 && Q > 0 && std::isfinite(P) && std::isfinite(Q))) return;
  const double a = p_total / P, b = q_total / Q;
  const double kl = (plogp - plogq) / P + a * std::log(Q / P);
  const double scaled = std::max(0.0, (kl - a * std::log(a / b)) / a);
  const double negative = b * std::sqrt(scaled / 2) + std::fabs(a - b);
  const double magnitude = std::fabs(kl) + 2 * negative;
  const double u = std::ldexp(1.0, -24), chain = static_cast<double>(c.width) + 3;
  const double margin = 1.05 * u * ((chain + 6) * magnitude + 10) + 1e-8;
  if (!std::isfinite(kl) || !std::isfinite(margin)) return;
  *lower = kl - margin;
  *upper = kl + margin;
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

// Threads for the passes of one call; they end with it.
class Search {
 public:
  explicit Search(size_t widest) : widest_(widest) {}
  ~Search() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : threads_) t.join();
  }
  // f(item, scratch) for items 0 ... n - 1, in blocks, on as many threads as are worth it
  template <typename F>
  void Run(size_t n, size_t block, F f) {
    const size_t want = std::min<size_t>(ThreadLimit(), n / block);
    next_ = 0;
    const std::function<void(Scratch*)> work = [&](Scratch* scratch) {
      try {
        for (size_t at = next_.fetch_add(block); at < n; at = next_.fetch_add(block))
          for (size_t i = at; i < std::min(n, at + block); ++i) f(i, scratch);
      } catch (...) {
        Fail(n);
      }
    };
    {
      std::lock_guard<std::mutex> lock(mutex_);
      work_ = &work;
      ++pass_;
      running_ = threads_.size();
    }
    wake_.notify_all();
    // the threads use this frame from here on: nothing leaves it before the last of them is done
    try {
      while (threads_.size() + 1 < want) {
        std::lock_guard<std::mutex> lock(mutex_);
        threads_.emplace_back(&Search::Loop, this, pass_ - 1);
        ++running_;
      }
    } catch (const std::exception&) {  // no more threads to be had: those that are there do
    }
    try {
      Scratch mine(widest_);
      work(&mine);
    } catch (...) {
      Fail(n);
    }
    std::unique_lock<std::mutex> lock(mutex_);
    done_.wait(lock, [&] { return running_ == 0; });
    if (failure_) std::rethrow_exception(failure_);
  }

 private:
  // keeps the exception in flight for Run's caller; no further items are taken
  void Fail(size_t n) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!failure_) failure_ = std::current_exception();
    next_ = n;
  }
  void Loop(size_t seen) {
    std::unique_ptr<Scratch> scratch;
    try {
      scratch.reset(new Scratch(widest_));
    } catch (const std::exception&) {  // takes no items: the other threads do them
    }
    std::unique_lock<std::mutex> lock(mutex_);
    while (true) {
      wake_.wait(lock, [&] { return stop_ || pass_ != seen; });
      if (stop_) return;
      seen = pass_;
      const std::function<void(Scratch*)>* const work = work_;
      lock.unlock();
      if (scratch) (*work)(scratch.get());
      lock.lock();
      if (--running_ == 0) done_.notify_all();
    }
  }
  const size_t widest_;
  std::vector<std::thread> threads_;
  std::mutex mutex_;
  std::condition_variable wake_, done_;
  const std::function<void(Scratch*)>* work_ = nullptr;  // of the Run in progress
  size_t pass_ = 0, running_ = 0;
  bool stop_ = false;
  std::atomic<size_t> next_{0};
  std::exception_ptr failure_;
};

}  // namespace

void CalibrateEntropyMany(size_t count, const float* const* hist, const float* const* hist_edges,
                          const size_t* num_bins, const int* num_quantized_bins,
                          const double* bounds, float* thresholds, float* divergences) {
  std::vector<Problem> problems;
  problems.reserve(count);
  size_t widest = 0;
  for (size_t i = 0; i < count; ++i) {
    problems.emplace_back(hist[i], hist_edges[i], num_bins[i], num_quantized_bins[i],
                          bounds == nullptr);
    widest = std::max(widest, num_bins[i]);
  }
  // neighbouring candidates in groups, the widest first
  struct Group {
    Problem* problem;
    long i;
    int count;
  };
  std::vector<Group> groups;
  for (Problem& p : problems)
    for (long i = p.zero_bin; i >= p.half; i -= kLanes)
      groups.push_back({&p, i, static_cast<int>(std::min<long>(kLanes, i - p.half + 1))});
  std::stable_sort(groups.begin(), groups.end(),
                   [](const Group& a, const Group& b) { return a.i > b.i; });
  Search search(widest);
  // every candidate's bounds, then the divergence of those that can be the smallest
  if (bounds != nullptr) {
    for (Problem& p : problems)
      for (size_t slot = 0; slot < p.candidates(); ++slot) {
        p.lower[slot] = *bounds++;
        p.upper[slot] = *bounds++;
      }
    groups.clear();
  }
  search.Run(groups.size(), 2, [&](size_t at, Scratch* scratch) {
    Problem& p = *groups[at].problem;
    const int count = groups[at].count;
    std::vector<Candidate> c;
    float take[kLanes] = {}, p_sum[kLanes] = {};
    Sums s[kLanes];
    bool smooth[kLanes];
    float* levels = scratch->levels.data();
    for (int l = 0; l < count; ++l) {
      c.emplace_back(p, groups[at].i - l);
      smooth[l] = Normalise(p, c[l], &s[l], levels + l * p.levels);
      take[l] = smooth[l] ? s[l].p_take : 0.f;
    }
    PSums(p, count, c.data(), take, p_sum);
    for (int l = 0; l < count; ++l) {
      if (!smooth[l]) continue;
      s[l].p_sum = p_sum[l];
      const size_t slot = groups[at].i - l - p.half;
      Estimate(p, c[l], s[l], levels + l * p.levels, &p.lower[slot], &p.upper[slot]);
    }
  });
  struct Item {
    Problem* problem;
    long i;
  };
  auto sum_up = [&](const std::vector<Item>& items) {
    search.Run(items.size(), 1, [&](size_t at, Scratch* scratch) {
      Problem& p = *items[at].problem;
      const Candidate c(p, items[at].i);
      Sums s;
      if (!Normalise(p, c, &s, scratch->levels.data())) return;
      PSums(p, 1, &c, &s.p_take, &s.p_sum);
      p.divergences[items[at].i - p.half] =
          Divergence(p, c, s, scratch->levels.data(), scratch);
    });
  };
  // First the one that promises the smallest: what it comes to rules out more of the others than
  // its upper bound.
  std::vector<Item> best, close;
  for (Problem& p : problems) {
    long at = -1;
    for (long i = p.half; i <= p.zero_bin; ++i) {
      const double low = p.lower[i - p.half], high = p.upper[i - p.half];
      if (std::isfinite(low) && std::isfinite(high) &&
          (at < 0 || low + high < p.lower[at - p.half] + p.upper[at - p.half]))
        at = i;
    }
    if (at >= 0) best.push_back({&p, at});
  }
  sum_up(best);
  for (Problem& p : problems) {
    const double smallest = *std::min_element(p.divergences.begin(), p.divergences.end());
    for (long i = p.zero_bin; i >= p.half; --i) {
      const double low = p.lower[i - p.half];
      if (low <= smallest && low < std::numeric_limits<double>::infinity() &&
          !(p.divergences[i - p.half] < std::numeric_limits<float>::infinity()))
        close.push_back({&p, i});
    }
  }
  sum_up(close);

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
  CalibrateEntropyMany(1, &hist, &hist_edges, &num_bins, &num_quantized_bins, nullptr, threshold,
                       divergence);
}

}  // namespace mxq_graph
