// The fully-connected kernels built for the requantized residual sum in the epilogue
// (mxq_quantized_fc_sum_requant).
#include "mxq_fc_kernels.h"

namespace mxq {

void fc_launch_sum_requant(hipStream_t s, const FcArgs& a, const FcLaunch& how,
                           const Workspace& ws) {
  fc_launch_mode<kEpiSumRq>(s, a, how, ws);
}

}  // namespace mxq
