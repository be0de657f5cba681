// Histogram of a float tensor over given bin edges: what the entropy calibration collects of
// every calibrated tensor (numpy.histogram in the reference's collector,
// python/mxnet/contrib/quantization.py:269-361), taken where the tensor lies instead of after
// a copy to the host.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mxq.h"
#include "mxq_common.h"

namespace mxq {
namespace {

constexpr int kThreads = 512;
// bins a work-group counts in LDS (64 KB); more are counted in memory directly
constexpr int kMaxLdsBins = 16384;

__global__ __launch_bounds__(kThreads) void zero_counts_kernel(uint32_t* counts, int bins) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < bins) counts[i] = 0;
}

// The equal-width formula only proposes a bin; the edges decide: bin k holds
// edges[k] <= x < edges[k + 1], the last one its upper edge as well, values outside the edges
// and NaN are left out (numpy corrects its own guess against the edges the same way, so the
// counts agree with it exactly).
// Bound by the LDS atomics and, at the end, one memory atomic per bin that a work-group filled:
// hence few work-groups with many values each (393216 values in 8001 bins: 1.45 ms on the host,
// copy included, 12 us here).
template <bool LDS>
__global__ __launch_bounds__(kThreads) void histogram_kernel(const float* __restrict__ in,
                                                             size_t n,
                                                             const float* __restrict__ edges,
                                                             int bins, uint32_t* counts) {
  extern __shared__ uint32_t local[];
  if (LDS) {
    for (int i = threadIdx.x; i < bins; i += kThreads) local[i] = 0;
    __syncthreads();
  }
  const float lo = edges[0], hi = edges[bins];
  const float per_unit = static_cast<float>(bins) / (hi - lo);
  const size_t stride = size_t(gridDim.x) * kThreads;
  for (size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride) {
    const float x = in[i];
    if (!(x >= lo && x <= hi)) continue;
    int k = static_cast<int>((x - lo) * per_unit);
    k = k < 0 ? 0 : k > bins - 1 ? bins - 1 : k;
    while (k > 0 && x < edges[k]) --k;
    while (k < bins - 1 && x >= edges[k + 1]) ++k;
    atomicAdd(LDS ? local + k : counts + k, 1u);
  }
  if (LDS) {
    __syncthreads();
    for (int i = threadIdx.x; i < bins; i += kThreads)
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
  // twice as many values as bins per work-group, so that counting outweighs the final atomics
  size_t grid = n / (lds ? 2 * static_cast<size_t>(bins) : kThreads) + 1;
  const size_t cap = static_cast<size_t>(num_cus()) * 2;
  if (grid > cap) grid = cap;
  if (lds)
    hipLaunchKernelGGL((histogram_kernel<true>), dim3(static_cast<unsigned>(grid)), dim3(kThreads),
                       static_cast<size_t>(bins) * sizeof(uint32_t), s, in, n, edges, bins,
                       counts);
  else
    hipLaunchKernelGGL((histogram_kernel<false>), dim3(static_cast<unsigned>(grid)),
                       dim3(kThreads), 0, s, in, n, edges, bins, counts);
  MXQ_LAUNCH_CHECK();
  MXQ_API_END();
}
