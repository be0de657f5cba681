// Histogram of a float tensor over given bin edges: what the entropy calibration collects of
// every calibrated tensor (numpy.histogram in the reference's collector,
// python/mxnet/contrib/quantization.py:269-361), taken where the tensor lies instead of after
// a copy to the host.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"

namespace mxq {
namespace {

constexpr int kThreads = 512;
// bins a work-group counts in LDS (64 KB, and their edges); more are counted in memory directly
constexpr int kMaxLdsBins = 16384;

__global__ __launch_bounds__(kThreads) void zero_counts_kernel(uint32_t* counts, int bins) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < bins) counts[i] = 0;
}

// The equal-width formula only proposes a bin; the edges decide: bin k holds
// edges[k] <= x < edges[k + 1], the last one its upper edge as well, values outside the edges
// and NaN are left out (numpy corrects its own guess against the edges the same way, so the
// counts agree with it exactly).
// Bound by latency: a value's load, its edges, its atomic.  So the edges lie in LDS beside the
// counts and a lane has eight values on their way; at the end there is one memory atomic per bin
// that a work-group filled, hence few work-groups with many values each.  196608 values in 8001
// bins 10 us; with the edges in memory and one value at a time 36, on the host 700.
// LDS: bins are counted there.  VALUES: of a lane in flight; with one, edges stay in memory.
// `holds`, where there is one, is 0 for edges that do not increase: between those a value would be
// moved on bin by bin through all of them, and nothing is counted.
template <bool LDS, int THREADS, int VALUES>
__global__ __launch_bounds__(THREADS) void histogram_kernel(const float* __restrict__ in, size_t n,
                                                            const float* __restrict__ edges,
                                                            int bins, uint32_t* counts,
                                                            const uint32_t* holds) {
  if (holds != nullptr && *holds == 0) return;
  constexpr bool HELD = VALUES > 1;  // the edges, in LDS
  extern __shared__ uint32_t local[];
  float* const edge_lds = reinterpret_cast<float*>(local + bins);
  const size_t stride = size_t(gridDim.x) * THREADS;
  size_t at = size_t(blockIdx.x) * THREADS + threadIdx.x;
  float x[VALUES];
  auto load = [&]() {
#pragma unroll
    for (int j = 0; j < VALUES; ++j) {
      const size_t i = at + j * stride;
      x[j] = i < n ? in[i] : NAN;
    }
    at += VALUES * stride;
  };
  load();
  if (LDS) {
    for (int i = threadIdx.x; i < bins; i += THREADS) local[i] = 0;
    if (HELD)
      for (int i = threadIdx.x; i <= bins; i += THREADS) edge_lds[i] = edges[i];
    __syncthreads();
  }
  const float* const e = HELD ? edge_lds : edges;
  const float lo = e[0], hi = e[bins];
  const float per_unit = static_cast<float>(bins) / (hi - lo);
  for (bool more = true; more;) {
    int k[VALUES];
    float low[VALUES], high[VALUES];
#pragma unroll
    for (int j = 0; j < VALUES; ++j) {
      const int guess = static_cast<int>((x[j] - lo) * per_unit);
      k[j] = guess < 0 ? 0 : guess > bins - 1 ? bins - 1 : guess;
      low[j] = e[k[j]];
      high[j] = e[k[j] + 1];
    }
#pragma unroll
    for (int j = 0; j < VALUES; ++j) {
      const float v = x[j];
      if (!(v >= lo && v <= hi)) continue;
      int b = k[j];
      if (v < low[j])
        while (b > 0 && v < e[b]) --b;
      else if (v >= high[j])
        while (b < bins - 1 && v >= e[b + 1]) ++b;
      atomicAdd(LDS ? local + b : counts + b, 1u);
    }
    more = at < n;
    if (more) load();
  }
  if (LDS) {
    __syncthreads();
    for (int i = threadIdx.x; i < bins; i += THREADS)
      if (local[i] != 0) atomicAdd(counts + i, local[i]);
  }
}

// The edges of `bins` equal bins over [-t, t], each as numpy computes it in float32 (index times
// step plus start, rounded twice; the last one t), and whether they increase and t is finite; the
// counts of the histogram that follows cleared.  t: the larger magnitude of range[0 ... 1], or `th`
// where that is no NaN; with `inside`, a range that reaches beyond it counts as one without edges.  (On
// the host the edges, their copy and a second wait for the device were half of what a tensor took.)
__global__ __launch_bounds__(1024) void symmetric_edges_kernel(const float* range, float th,
                                                               bool inside, int bins, float* edges,
                                                               uint32_t* increase,
                                                               uint32_t* counts) {
  const float x = fabsf(range[0]), y = fabsf(range[1]), reach = (x < y) ? y : x;
  const float t = th != th ? reach : th;
  const float step = (t + t) / static_cast<float>(bins);
  bool ok = t < INFINITY && !(inside && reach > t);
  for (int i = threadIdx.x; i < bins; i += 1024) {
    const float edge = static_cast<float>(i) * step - t;
    const float next = i + 1 < bins ? static_cast<float>(i + 1) * step - t : t;
    ok = ok && next > edge;
    edges[i] = edge;
    counts[i] = 0;
  }
  if (threadIdx.x == 0) edges[bins] = t;
  ok = __syncthreads_and(ok) != 0;
  if (threadIdx.x == 0) *increase = ok;
}

void launch_histogram(hipStream_t s, const float* in, size_t n, const float* edges, int bins,
                      uint32_t* counts, const uint32_t* holds) {
  if (n == 0) return;
  const bool lds = bins <= kMaxLdsBins;
  // Eight values a lane and the edges in LDS where there are values for them (us, one value / eight:
  // 100 values 4.4 / 4.9, 1000 in 101 bins 4.4 / 4.9, in 1001 5.2 / 5.1, 10000 in 11 bins 4.6 / 5.7, in
  // 101 4.7 / 5.1, in 1001 6.2 / 5.4, 100000 in 11 6.5 / 6.1, in 8001 19.3 / 9.3).  Counted in memory there
  // is nothing to win (10000 in 20001 bins 5.4 / 7.6, 1000000 50.7 / 51.3).
  const bool eight = lds && (n >= 65536 || (n >= 1536 && bins >= 512));
  const int threads = eight ? 1024 : 512;
  // twice as many values as bins per work-group, so that counting outweighs the final atomics
  size_t grid = n / (lds ? 2 * static_cast<size_t>(bins) : threads) + 1;
  const size_t cap = static_cast<size_t>(num_cus()) * (bins <= kMaxLdsBins / 2 || !eight ? 2 : 1);
  if (grid > cap) grid = cap;
  const size_t words = lds ? (eight ? 2 * static_cast<size_t>(bins) + 1 : bins) : 0;
  const auto kernel = eight ? histogram_kernel<true, 1024, 8>
                            : lds ? histogram_kernel<true, 512, 1> : histogram_kernel<false, 512, 1>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(threads),
                     words * sizeof(uint32_t), s, in, n, edges, bins, counts, holds);
  MXQ_LAUNCH_CHECK();
}

}  // namespace
}  // namespace mxq

using namespace mxq;

static int symmetric_histogram(void* stream, const float* in, size_t n, int bins, float th,
                               bool inside, uint32_t* out, void* workspace,
                               size_t workspace_bytes) {
  MXQ_API_BEGIN();
  MXQ_CHECK(bins > 0 && bins <= (1 << 24), "a histogram needs at least one bin, and at most 2^24");
  MXQ_CHECK(n > 0 && n <= 0xffffffffu, "counts are 32 bits wide, and no value has no range");
  MXQ_CHECK(in != nullptr && out != nullptr && workspace != nullptr, "null pointer");
  const size_t extremes = mxq_minmax_f32_workspace(n);
  MXQ_CHECK(workspace_bytes >= mxq_symmetric_histogram_f32_workspace(n, bins) &&
                (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0,
            "workspace too small or unaligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* const ws = static_cast<char*>(workspace);
  float* const range = reinterpret_cast<float*>(out);
  float* const edges = reinterpret_cast<float*>(ws + extremes);
  const int status = mxq_minmax_f32(stream, in, n, range, range + 1, ws, extremes);
  if (status != 0) return status;
  hipLaunchKernelGGL(symmetric_edges_kernel, dim3(1), dim3(1024), 0, s, range, th, inside, bins,
                     edges, out + 2, out + 3);
  MXQ_LAUNCH_CHECK();
  launch_histogram(s, in, n, edges, bins, out + 3, out + 2);
  MXQ_API_END();
}

extern "C" {

int mxq_histogram_f32(void* stream, const float* in, size_t n, const float* edges, int bins,
                      uint32_t* counts) {
  MXQ_API_BEGIN();
  MXQ_CHECK(bins > 0, "a histogram needs at least one bin");
  MXQ_CHECK(n <= 0xffffffffu, "counts are 32 bits wide");
  MXQ_CHECK(edges != nullptr && counts != nullptr && (n == 0 || in != nullptr), "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(zero_counts_kernel, dim3((bins + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     s, counts, bins);
  MXQ_LAUNCH_CHECK();
  if (n == 0) return 0;
  launch_histogram(s, in, n, edges, bins, counts, nullptr);
  MXQ_API_END();
}

size_t mxq_symmetric_histogram_f32_workspace(size_t n, int bins) {
  return (static_cast<size_t>(bins > 0 ? bins : 0) * 4 + 4 + 255) / 256 * 256 +
         mxq_minmax_f32_workspace(n);
}

int mxq_symmetric_histogram_f32(void* stream, const float* in, size_t n, int bins, float th,
                                uint32_t* out, void* workspace, size_t workspace_bytes) {
  return symmetric_histogram(stream, in, n, bins, th, false, out, workspace, workspace_bytes);
}

int mxq_symmetric_histogram_inside_f32(void* stream, const float* in, size_t n, int bins, float th,
                                       uint32_t* out, void* workspace, size_t workspace_bytes) {
  return symmetric_histogram(stream, in, n, bins, th, true, out, workspace, workspace_bytes);
}

}  // extern "C"
