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
template <bool LDS, int THREADS, int VALUES>
__global__ __launch_bounds__(THREADS) void histogram_kernel(const float* __restrict__ in, size_t n,
                                                            const float* __restrict__ edges,
                                                            int bins, uint32_t* counts) {
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

}  // namespace
}  // namespace mxq

using namespace mxq;

extern "C" int mxq_histogram_f32(void* stream, const float* in, size_t n, const float* edges,
                                 int bins, uint32_t* counts) {
  MXQ_API_BEGIN();
  MXQ_CHECK(bins > 0, "a histogram needs at least one bin");
  MXQ_CHECK(n <= 0xffffffffu, "counts are 32 bits wide");
  MXQ_CHECK(edges != nullptr && counts != nullptr && (n == 0 || in != nullptr), "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(zero_counts_kernel, dim3((bins + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     s, counts, bins);
  MXQ_LAUNCH_CHECK();
  if (n == 0) return 0;
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
                     words * sizeof(uint32_t), s, in, n, edges, bins, counts);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}
