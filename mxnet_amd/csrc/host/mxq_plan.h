// A network's forward pass as a list of launches with resolved shapes: what executor.py's
// planner (_plan.py) makes of a quantized graph, and what one Executor.forward runs.
//
// Activations live in one arena per call, taken from torch's caching allocator and given back
// when the call returns (stream order keeps the memory valid for the launches), at offsets the
// planner assigned from their lifetimes; weights and constant ranges are device tensors that the
// plan holds.  The launches of a plan are immutable once built and it may run from several threads
// and streams.
#ifndef MXQ_PLAN_H_
#define MXQ_PLAN_H_

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../../include/mxq_ops.h"

namespace mxq_plan {

// Where an operand lies.
struct Ref {
  enum Base : int { kNull = 0, kArena = 1, kHeld = 2, kFeed = 3, kOutput = 4 };
  int base = kNull;
  int index = 0;       // of the held tensor, feed or output
  int64_t offset = 0;  // bytes
};

enum class Kind : int {
  kNode,         // any registered operator
  kConv,         // convolution -> requantize (-> relu), NHWC
  kFc,           // fully connected -> requantize (-> relu)
  kFcF32,        // fully connected -> requantize -> dequantize
  kFcSum,        // ... -> requantize -> sum over a calibrated range (-> relu)
  kFcSumRq,      // ... -> requantize -> sum -> requantize (-> relu)
  kQuantNhwc,    // calibrated quantize of a float image into NHWC
  kToNhwc,       // int8 NCHW -> NHWC, channels padded
  kFromNhwc,     // back
  kPool,         // NHWC pooling
  kRelu,         // int8 relu
  kAdd,          // int8 sum, int32 or calibrated int8
  kRequantize,   // calibrated
  kBlock,        // 3 x 3 convolution -> 1 x 1 -> sum (-> 1 x 1), each requantized
  kConvPair,     // two 1 x 1 convolutions of one tensor, each requantized (-> relu)
  kConvPool,     // 4 x 4 convolution, requantized (-> relu) -> 3 x 3 maximum
  kConv3x3,      // 3 x 3 convolution over many channels, requantized (-> relu)
};

struct Step {
  Kind kind;
  std::vector<int64_t> ints;
  std::vector<float> floats;
  std::vector<Ref> refs;
  void* node = nullptr;          // kNode
  std::vector<mxq_blob> blobs;   // kNode: inputs, then outputs; `data` is filled per call
  int num_in = 0;
};

struct Output {
  std::vector<int64_t> shape;
  at::ScalarType type;
};

struct Plan {
  int64_t arena_bytes = 0;
  std::vector<at::Tensor> held;
  std::vector<Step> steps;
  std::vector<Output> outputs;
  int device = 0;
  // that the allocator knows of for the held tensors: the one that built the plan, and those that
  // it has run on since
  std::vector<c10::hip::HIPStream> streams;

  // To be called before launches on `stream`, under the interpreter lock.  The held tensors come
  // from the stream that built the plan (or from the caller): the allocator is told of every other
  // stream that reads them, once for each, so that memory of a plan that is dropped with launches
  // pending there is not given away before they end.  (0.8 us a tensor; 400 of them in a quantized
  // ResNet-50.)
  void used_on(c10::hip::HIPStream stream);

  // Enqueues every step on `stream`; false: *error says what failed.
  bool run(void* stream, const std::vector<at::Tensor>& feeds,
           const std::vector<at::Tensor>& outs, const at::Tensor& arena, std::string* error) const;
};

}  // namespace mxq_plan

#endif  // MXQ_PLAN_H_
