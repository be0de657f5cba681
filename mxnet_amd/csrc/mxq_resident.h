// The 1 x 1 convolution / fully-connected kernel whose weights stay in registers
// (mxq_resident.hip): its arguments, its launcher and the rule that chooses it.
#ifndef MXQ_RESIDENT_H_
#define MXQ_RESIDENT_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "mxq_gemm.h"

namespace mxq {

struct ResidentArgs {
  const int8_t* data;    // [M][K], or NHWC images of a strided 1 x 1 convolution
  const int8_t* weight;  // [N][K]
  int M, N, K;
  int ldo;               // output row pitch in elements
  Epilogue epi;          // out8 alone
  // strided convolution only (area = 0: rows of K bytes one behind the other)
  int area, OW;          // output pixels per image, and per line
  long long image;       // bytes between images
  int down, right;       // bytes between the pixels of two output lines, of two output columns
  int images;
};

// Whether the kernel takes the launch, and is the faster one.  `aligned`: 16-byte aligned operands
// and output.
bool resident_wins(const ResidentArgs& a, bool aligned);
void launch_resident(hipStream_t s, const ResidentArgs& a);
// Two layers over the same rows in one launch.
bool resident_pair_wins(const ResidentArgs& a, const ResidentArgs& b, bool aligned);
void launch_resident_pair(hipStream_t s, const ResidentArgs& a, const ResidentArgs& b);

}  // namespace mxq
#endif  // MXQ_RESIDENT_H_
