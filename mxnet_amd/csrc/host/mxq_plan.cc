// The launches of a plan (mxq_plan.h).
#include "mxq_plan.h"

#include "../../../include/mxq.h"

namespace mxq_plan {

void Plan::used_on(c10::hip::HIPStream stream) {
  for (const auto& s : streams)
    if (s == stream) return;
  // tensors of this build name the device type CUDA
  const c10::Stream named(c10::Stream::UNSAFE,
                          c10::Device(c10::DeviceType::CUDA, stream.device_index()), stream.id());
  for (const at::Tensor& t : held) t.record_stream(named);
  streams.push_back(stream);
}

bool Plan::run(void* stream, const std::vector<at::Tensor>& feeds,
               const std::vector<at::Tensor>& outs, const at::Tensor& arena,
               std::string* error) const {
  char* base = arena.defined() ? static_cast<char*>(arena.data_ptr()) : nullptr;
  auto at = [&](const Ref& r) -> void* {
    switch (r.base) {
      case Ref::kArena: return base + r.offset;
      case Ref::kHeld: return static_cast<char*>(held[r.index].data_ptr()) + r.offset;
      case Ref::kFeed: return static_cast<char*>(feeds[r.index].data_ptr()) + r.offset;
      case Ref::kOutput: return static_cast<char*>(outs[r.index].data_ptr()) + r.offset;
      default: return nullptr;
    }
  };
  std::vector<mxq_blob> blobs;
  for (const Step& s : steps) {
    const int64_t* n = s.ints.data();
    const float* f = s.floats.data();
    auto p = [&](int i) { return at(s.refs[i]); };
    auto q = [&](int i) { return static_cast<int8_t*>(at(s.refs[i])); };
    auto v = [&](int i) { return static_cast<float*>(at(s.refs[i])); };
    auto i = [&](int k) { return static_cast<int>(n[k]); };
    int rc = 0;
    switch (s.kind) {
      case Kind::kNode: {
        blobs = s.blobs;
        for (size_t k = 0; k < blobs.size(); ++k) blobs[k].data = p(static_cast<int>(k));
        rc = mxq_node_forward(s.node, stream, device, s.num_in, blobs.data(),
                              static_cast<int>(blobs.size()) - s.num_in, blobs.data() + s.num_in,
                              p(static_cast<int>(blobs.size())), static_cast<size_t>(n[0]));
        if (rc != 0) {
          *error = mxq_ops_last_error();
          return false;
        }
        continue;
      }
      // refs: data, weight, bias, six ranges, scratch, output, workspace[, residual, its
      // range[, pairs]], what mxq_prepare_layer made of bias and ranges where those stay
      case Kind::kConv:
        if (const void* prepared = at(s.refs.back()))
          rc = mxq_quantized_conv_nhwc_prepared(
              stream, q(0), q(1), prepared, i(0), i(1), i(2), i(3), i(4), i(5), i(6), i(7), i(8),
              i(9), i(10), i(11), i(12), q(10), i(13), f[0], f[1], p(11),
              static_cast<size_t>(n[14]));
        else
          rc = mxq_quantized_conv_nhwc(
              stream, q(0), q(1), q(2), i(0), i(1), i(2), i(3), i(4), i(5), i(6), i(7), i(8), i(9),
              i(10), i(11), i(12), v(3), v(4), v(5), v(6), v(7), v(8), nullptr, v(9), v(9) + 1,
              q(10), v(9) + 2, v(9) + 3, i(13), f[0], f[1], p(11), static_cast<size_t>(n[14]));
        break;
      case Kind::kFc:
      case Kind::kFcF32: {
        const bool floats = s.kind == Kind::kFcF32;
        if (const void* prepared = at(s.refs.back()))
          rc = mxq_quantized_fc_prepared(stream, q(0), q(1), prepared, i(0), i(1), i(2),
                                         floats ? nullptr : q(10), floats ? v(10) : nullptr, i(3),
                                         f[0], f[1], p(11), static_cast<size_t>(n[4]));
        else if (floats)
          rc = mxq_quantized_fc_f32(stream, q(0), q(1), q(2), i(0), i(1), i(2), v(3), v(4), v(5),
                                    v(6), v(7), v(8), v(10), v(9), v(9) + 1, v(9) + 2, v(9) + 3,
                                    i(3), f[0], f[1], p(11), static_cast<size_t>(n[4]));
        else
          rc = mxq_quantized_fc(stream, q(0), q(1), q(2), i(0), i(1), i(2), v(3), v(4), v(5), v(6),
                                v(7), v(8), nullptr, v(9), v(9) + 1, q(10), v(9) + 2, v(9) + 3,
                                i(3), f[0], f[1], p(11), static_cast<size_t>(n[4]));
        break;
      }
      case Kind::kFcSum:
      case Kind::kFcSumRq: {
        const bool requant = s.kind == Kind::kFcSumRq;
        const void* pairs = requant ? p(15) : nullptr;
        if (const void* prepared = at(s.refs.back()))
          rc = mxq_quantized_fc_sum_prepared(
              stream, q(0), q(1), prepared, i(0), i(1), i(2), q(12), v(13), v(14), q(10), f[0],
              f[1], f[2], f[3], i(3), requant, pairs, p(11), static_cast<size_t>(n[4]));
        else if (requant)
          rc = mxq_quantized_fc_sum_requant(
              stream, q(0), q(1), q(2), i(0), i(1), i(2), v(3), v(4), v(5), v(6), v(7), v(8),
              q(12), v(13), v(14), q(10), v(9), v(9) + 1, v(9) + 2, v(9) + 3, f[0], f[1], f[2],
              f[3], i(3), pairs, p(11), static_cast<size_t>(n[4]));
        else
          rc = mxq_quantized_fc_sum(stream, q(0), q(1), q(2), i(0), i(1), i(2), v(3), v(4), v(5),
                                    v(6), v(7), v(8), q(12), v(13), v(14), q(10), v(9), v(9) + 1,
                                    v(9) + 2, v(9) + 3, f[0], f[1], f[2], f[3], i(3), p(11),
                                    static_cast<size_t>(n[4]));
        break;
      }
      case Kind::kQuantNhwc:
        if (i(5))
          rc = mxq_quantize_to_s2d(stream, v(0), q(1), v(2), v(2) + 1, i(0), i(1), i(2), i(3),
                                   i(4), i(6), i(7), i(8), i(9), f[0], f[1]);
        else
          rc = mxq_quantize_to_nhwc(stream, v(0), q(1), v(2), v(2) + 1, i(0), i(1), i(2), i(3),
                                    i(4), 0, 0, 0, f[0], f[1]);
        break;
      case Kind::kToNhwc:
        rc = mxq_nchw_to_nhwc_pad_i8(stream, q(0), q(1), i(0), i(1), i(2), i(3), i(4));
        break;
      case Kind::kFromNhwc:
        rc = mxq_nhwc_pad_to_nchw_i8(stream, q(0), q(1), i(0), i(1), i(2), i(3), i(4));
        break;
      case Kind::kPool:
        rc = mxq_quantized_pooling_nhwc(stream, q(0), i(0), i(1), i(2), i(3), i(4), i(5), i(6),
                                        i(7), i(8), i(9), i(10), i(11), i(12), i(13), q(1));
        break;
      case Kind::kRelu:
        rc = mxq_quantized_relu(stream, q(0), v(2), v(3), q(1), v(4), v(4) + 1,
                                static_cast<size_t>(n[0]));
        break;
      case Kind::kAdd:  // refs: lhs, rhs, output, four ranges, output range
        rc = mxq_quantized_elemwise_add(stream, p(0), MXQ_INT8, p(1), MXQ_INT8, v(3), v(4), v(5),
                                        v(6), p(2), i(1), v(7), v(7) + 1,
                                        static_cast<size_t>(n[0]), i(2), f[0], f[1]);
        break;
      case Kind::kBlock:  // refs: data, weights, what mxq_prepare_block made, what
                          // mxq_prepare_layer made of three layers, residual, sum, third output
        rc = mxq_quantized_block(stream, q(0), q(1), p(2), p(3), p(4), p(5), i(0), i(1), i(2),
                                 i(3), i(4), i(5), i(6), q(6), q(7), q(8), i(7), i(8));
        break;
      case Kind::kConvPair:  // refs: data, both weights, outputs, what mxq_prepare_layer made
        rc = mxq_quantized_conv_pair_prepared(stream, q(0), i(0), i(1), i(2), i(3), i(6), i(7),
                                              q(1), p(5), i(4), q(3), i(8), f[0], f[1], q(2), p(6),
                                              i(5), q(4), i(9), f[2], f[3]);
        break;
      case Kind::kConvPool:  // refs: data, weights, what mxq_prepare_layer made, output
        rc = mxq_quantized_conv_pool(stream, q(0), q(1), p(2), i(0), i(1), i(2), i(3), i(4), i(5),
                                     i(6), i(7), i(8), i(9), i(10), q(3), i(11));
        break;
      case Kind::kConv3x3:  // refs: data, weights, what mxq_prepare_layer made, output
        rc = mxq_quantized_conv3x3(stream, q(0), q(1), p(2), i(0), i(1), i(2), i(3), i(4), q(3),
                                   i(5));
        break;
      case Kind::kRequantize:
        rc = mxq_requantize(stream, static_cast<int32_t*>(p(0)), v(2), v(3), q(1), v(4), v(4) + 1,
                            static_cast<size_t>(n[0]), 1, f[0], f[1], nullptr, 0);
        break;
    }
    if (rc != 0) {
      *error = mxq_last_error();
      return false;
    }
  }
  return true;
}

}  // namespace mxq_plan
