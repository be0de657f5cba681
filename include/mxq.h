/*
 * mxq.h - C ABI of libmxq_hip.so: MI355X (gfx950) kernels for MXNet's INT8
 * quantized-inference operators.
 *
 * This is the launcher the C++ FCompute<gpu> host functions call in place of
 * mshadow's Kernel<OP,gpu>::Launch, broadcast::RTCReduce, cublasGemmEx and
 * cudnnConvolutionForward.  Every entry point
 *   - takes plain device pointers, sizes and a raw hipStream_t (as void*; NULL
 *     is the default stream),
 *   - only enqueues work on that stream: no allocation, no free, no device or
 *     stream synchronisation, no retained state (the library has no mutable
 *     process-wide variables; the entry points are re-entrant and may be called
 *     concurrently from different threads on different streams, provided that
 *     calls in flight at the same time do not share a workspace),
 *   - returns 0 on success and -1 on failure with the message available from
 *     mxq_last_error() on the calling thread (the convention of
 *     include/mxnet/c_api_error.h:39-58 in the reference).
 * All pointers named min / max are DEVICE pointers to one float32, exactly as the
 * reference's min/max TBlobs of shape (1,).
 *
 * Reference paths are relative to the apache/mxnet tree.
 */
#ifndef MXQ_H_
#define MXQ_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MXQ_ABI_VERSION 3

/* element type codes = mshadow::TypeFlag (3rdparty/mshadow/mshadow/base.h:351-364) */
#define MXQ_FLOAT32 0
#define MXQ_FLOAT64 1
#define MXQ_UINT8 3
#define MXQ_INT32 4
#define MXQ_INT8 5
#define MXQ_INT64 6

/* Last error message of the calling thread ("" if none). */
const char* mxq_last_error(void);
int mxq_abi_version(void);

/* ---- _contrib_quantize_v2 ------------------------------------------------
 * Replaces QuantizeV2Operator<gpu>::Forward for fp32 input
 * (src/operator/quantization/quantize_v2-inl.h:218-305): the
 * Kernel<quantize_v2_zero_centered|quantize_v2_unsigned,gpu>::Launch calls and,
 * when uncalibrated, the two broadcast::RTCReduce passes (min, max) in front
 * of them.  out_type is MXQ_INT8 or MXQ_UINT8 (the reference's GPU build
 * refuses uint8, :198-201; here it follows the CPU kernel :66-95 and
 * saturates where the reference is undefined).  calibrated != 0 uses
 * (min_calib, max_calib); otherwise the range is reduced on the device in
 * `workspace` (>= mxq_quantize_v2_workspace(n) bytes, 16-byte aligned) and
 * never crosses the host. */
size_t mxq_quantize_v2_workspace(size_t n);
int mxq_quantize_v2(void* stream, const float* in, void* out, float* omin, float* omax,
                    size_t n, int out_type, int calibrated, float min_calib, float max_calib,
                    void* workspace, size_t workspace_bytes);

/* mxq_quantize_v2 for callers that cannot allocate (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc) and bring no workspace: the reduction
 * partials of the uncalibrated path live in a 16 KiB array inside the library's device
 * image (one copy per GPU, held until the process ends).  It has no counterpart in the
 * reference, whose operator always draws its temp space from the framework's resource
 * pool.  Same arguments and results as mxq_quantize_v2 without the workspace; n is
 * limited to 2^31 elements (a larger n is refused with an error).  The call allocates and
 * frees nothing.  All calls on one GPU share that GPU's array: calls that overlap in time
 * on one GPU (different streams) race on it and must be serialised by the caller; calls
 * on one stream, or on different GPUs, are safe.  The first uncalibrated call on a GPU
 * looks the array's address up (hipGetDevice, hipGetSymbolAddress: host runtime calls that
 * may load the code object); make that first call outside any stream capture, every later
 * call on that GPU only launches kernels and may be captured. */
int mxq_quantize_v2_noalloc(void* stream, const float* in, void* out, float* omin, float* omax,
                            size_t n, int out_type, int calibrated, float min_calib,
                            float max_calib);

/* ---- _contrib_quantize (v1) ---------------------------------------------
 * Replaces QuantizeCompute<gpu> (src/operator/quantization/quantize-inl.h:90-131):
 * same kernels, the range arrives as two device scalars. */
int mxq_quantize(void* stream, const float* in, const float* imin, const float* imax, void* out,
                 float* omin, float* omax, size_t n, int out_type);

/* Identity pass for int8/uint8 input of quantize_v2 (quantize_v2-inl.h:203-216):
 * copies n bytes and writes the constant ranges. */
int mxq_quantize_v2_passthrough(void* stream, const void* in, void* out, float* omin,
                                float* omax, size_t n, int in_type, int calibrated,
                                float min_calib, float max_calib);

/* ---- _contrib_requantize -------------------------------------------------
 * Replaces RequantizeForward<gpu> (src/operator/quantization/requantize-inl.h:127-240):
 * int32 -> int8 with the input range (imin, imax) read from the device;
 * calibrated uses MaxAbs(min_calib, max_calib), uncalibrated reduces the int32
 * min and max on the device first (workspace as above). */
size_t mxq_requantize_workspace(size_t n);
int mxq_requantize(void* stream, const int32_t* in, const float* imin, const float* imax,
                   int8_t* out, float* omin, float* omax, size_t n, int calibrated,
                   float min_calib, float max_calib, void* workspace, size_t workspace_bytes);

/* ---- _contrib_dequantize -------------------------------------------------
 * Replaces DequantizeOperator<gpu>::Forward
 * (src/operator/quantization/dequantize-inl.h:115-144); in_type MXQ_INT8 or
 * MXQ_UINT8. */
int mxq_dequantize(void* stream, const void* in, int in_type, const float* imin,
                   const float* imax, float* out, size_t n);

/* ---- _contrib_quantized_act (relu) -----------------------------------------
 * int8 max(x, 0); the range passes through unchanged
 * (src/operator/quantization/quantized_activation.cc:84-120, CPU-only in the
 * reference through dnnl/dnnl_quantized_act.cc:33-45). */
int mxq_quantized_relu(void* stream, const int8_t* in, const float* imin, const float* imax,
                       int8_t* out, float* omin, float* omax, size_t n);

/* ---- _contrib_quantized_pooling ---------------------------------------------
 * Replaces QuantizedCuDNNPoolingOp::Forward
 * (src/operator/quantization/quantized_pooling.cu:33-128): cudnnPoolingForward on
 * the NCHW int8 tensor plus the two range copies.  OH / OW are the extents
 * QuantizedPoolingShape computed (quantized_pooling.cc:82-121; global pooling is
 * kernel = (H, W), stride 1, OH = OW = 1).  Windows and the divisor of avg follow
 * the reference's own pooling loops (src/operator/nn/pool.h:476-522):
 * count_include_pad != 0 is cuDNN's COUNT_INCLUDE_PADDING, the mode the reference
 * selects.  max ignores padding; avg returns nearest-even(sum / divisor): that
 * rounding lives inside cuDNN / oneDNN in the reference and is not pinned by its
 * sources (its test accepts +-2).  in_type MXQ_INT8 or MXQ_UINT8 (the reference's
 * GPU build takes int8 only). */
#define MXQ_POOL_MAX 0
#define MXQ_POOL_AVG 1
int mxq_quantized_pooling_nchw(void* stream, const void* in, int in_type, int N, int C, int H,
                               int W, int kernel_h, int kernel_w, int stride_h, int stride_w,
                               int pad_h, int pad_w, int OH, int OW, int pool_type,
                               int count_include_pad, const float* imin, const float* imax,
                               void* out, float* omin, float* omax);

/* ---- _contrib_quantized_flatten ----------------------------------------------
 * Replaces QuantizedFlattenCompute (src/operator/quantization/quantized_flatten-inl.h:39-94;
 * registered for cpu only in the reference, quantized_flatten.cc:35): copies n_bytes
 * of int8/uint8 data and the two range scalars; in == out (the operator's in-place
 * option, quantized_flatten.cc:52-56) copies nothing. */
int mxq_quantized_flatten(void* stream, const void* in, const float* imin, const float* imax,
                          void* out, float* omin, float* omax, size_t n_bytes);

/* ---- _contrib_quantized_elemwise_add ---------------------------------------------
 * Replaces DNNLQuantizedElemwiseAddForward
 * (src/operator/quantization/dnnl/dnnl_quantized_elemwise_add.cc:134-257; the operator is
 * cpu-only in the reference, quantized_elemwise_add.cc:80-87) for operands of one shape:
 * out = saturate(nearest-even(lhs * s0 + rhs * s1)) in binary32, s = output scale / input
 * scale with the reference's ranges (127.5 int8, 255.5 uint8, 2^31 - 1 int32).
 * Uncalibrated: out is int32 over (-(|A|+|B|), |A|+|B|).  Calibrated: out has the inputs'
 * type (int8 when they differ) over (min_calib, max_calib).  A uint8 operand beside an
 * int8 one is first halved to int8, as the reference does.  The rounding itself lives
 * inside oneDNN in the reference and is not pinned by its sources (its test accepts a
 * dequantized error of 2). */
int mxq_quantized_elemwise_add(void* stream, const void* lhs, int lhs_type, const void* rhs,
                               int rhs_type, const float* lhs_min, const float* lhs_max,
                               const float* rhs_min, const float* rhs_max, void* out, int out_type,
                               float* omin, float* omax, size_t n, int calibrated,
                               float min_calib, float max_calib);

/* _contrib_quantized_npi_add (src/operator/quantization/quantized_elemwise_add.cc:141-178,
 * dnnl/dnnl_quantized_elemwise_add.cc:134-257; cpu only in the reference): the quantized sum
 * of two contiguous operands under numpy broadcasting (shapes aligned at the last axis, an
 * extent of 1 stretches).  Equal shapes are forwarded to mxq_quantized_elemwise_add; for
 * different shapes a uint8 operand next to an int8 one is taken at its own scale, as the
 * reference's binary primitive does.  out_type as for mxq_quantized_elemwise_add; the output
 * has fewer than 2^32 elements. */
int mxq_quantized_broadcast_add(void* stream, const void* lhs, int lhs_type, int lhs_ndim,
                                const int64_t* lhs_shape, const void* rhs, int rhs_type,
                                int rhs_ndim, const int64_t* rhs_shape, const float* lhs_min,
                                const float* lhs_max, const float* rhs_min, const float* rhs_max,
                                void* out, int out_type, float* omin, float* omax,
                                int calibrated, float min_calib, float max_calib);

/* ---- _contrib_quantized_elemwise_mul ---------------------------------------------
 * Replaces QuantizedElemwiseMulOpForward
 * (src/operator/quantization/quantized_elemwise_mul.cc:114-206; registered for cpu only,
 * :232) for int8 operands of one shape: out[i] = (out_type)(lhs[i] * rhs[i] * out_scale),
 * the int product converted to binary32, multiplied, truncated.
 *   out_type MXQ_INT32 (uncalibrated): out_scale = 1, range from
 *     QuantizationRangeForMultiplication<int8,int8,int32> (quantization_utils.h:141-170);
 *   out_type MXQ_INT8 (calibrated): out_scale = (127.5 / MaxAbs(calib)) / lhs_scale /
 *     rhs_scale with scale = 127.5 / MaxAbs(range), range (min_calib, max_calib);
 *   out_type MXQ_FLOAT32 (enable_float_output): out_scale = 1 / lhs_scale / rhs_scale in
 *     binary64, rounded once; omin / omax are not written and may be NULL.
 * A calibrated product whose truncated value does not fit int8 is undefined in the
 * reference; the low byte of the truncated int32 is stored (what its x86 build does). */
int mxq_quantized_elemwise_mul(void* stream, const int8_t* lhs, const int8_t* rhs,
                               const float* lhs_min, const float* lhs_max, const float* rhs_min,
                               const float* rhs_max, void* out, int out_type, float* omin,
                               float* omax, size_t n, int calibrated, float min_calib,
                               float max_calib);

/* ---- _contrib_quantized_embedding --------------------------------------------------
 * Replaces QuantizedEmbeddingOpForward
 * (src/operator/quantization/quantized_indexing_op.cc:103-122; cpu only, :146) and the
 * TakeZeroAxisCPU<clip> kernel it launches (src/operator/tensor/indexing_op.cc:30-61):
 * out[i, :] = weight[clip(int64(indices[i]), 0, input_dim - 1), :], int8 rows of output_dim
 * bytes; the weight's range is passed through.  index_type is the mshadow type flag of
 * `indices` (float32, float64, uint8, int32, int8 or int64). */
int mxq_quantized_embedding(void* stream, const void* indices, int index_type,
                            const int8_t* weight, const float* min_weight,
                            const float* max_weight, int8_t* out, float* omin, float* omax,
                            size_t n_indices, int64_t input_dim, int64_t output_dim);

/* ---- _contrib_quantized_transpose --------------------------------------------------
 * Replaces DNNLQuantizedTransposeForward
 * (src/operator/quantization/dnnl/dnnl_quantized_transpose.cc; shapes and types
 * quantized_transpose.cc:31-66; cpu only in the reference): out = in permuted so that out
 * axis d is in axis axes[d] (axes == NULL reverses the axes, TransposeParam's default),
 * one byte per element (int8 or uint8), ndim <= 8; the range is passed through.
 * _contrib_quantized_reshape (quantized_reshape.cc:31-46) needs no entry point of its own:
 * it is mxq_quantized_flatten's copy. */
int mxq_quantized_transpose(void* stream, const void* in, const float* imin, const float* imax,
                            void* out, float* omin, float* omax, int ndim,
                            const int64_t* in_shape, const int* axes);

/* ---- _contrib_quantize_asym ----------------------------------------------------------
 * Replaces QuantizeAsymOp<gpu>::Forward
 * (src/operator/quantization/quantize_asym-inl.h:78-160): float32 -> uint8 with
 * scale = 255 / (max - min), shift = 255 - max * scale,
 * out = (uint8)(in * scale + shift + 0.5) (the 0.5 in binary64), over (min_calib,
 * max_calib) or, uncalibrated, the data's own min and max (workspace of
 * mxq_quantize_asym_workspace(n) bytes, 16-byte aligned).  int8 input: out = in + 128,
 * scale 1, shift 128; uint8 input: copied, scale 1, shift 0.  A value outside [0, 256) is
 * undefined in the reference; the low byte of the truncated int32 is stored. */
size_t mxq_quantize_asym_workspace(size_t n);
int mxq_quantize_asym(void* stream, const void* in, int in_type, uint8_t* out, float* oscale,
                      float* oshift, size_t n, int calibrated, float min_calib, float max_calib,
                      void* workspace, size_t workspace_bytes);

/* ---- _contrib_quantized_batch_norm, _contrib_quantized_batch_norm_relu ----------------
 * Replaces DNNLQuantizedBatchNormForward
 * (src/operator/quantization/dnnl/dnnl_quantized_batch_norm.cc:34-130; cpu-only in the
 * reference): data [outer][channels][inner] int8 (uint8 is first scaled to int8 by
 * 127.5 / 255.5), inference statistics.  Per channel
 *   invstd = float(1.0 / sqrt(double(var) + eps)),
 *   w = gamma * invstd * MaxAbs(data range) / MaxAbs(calib range),
 *   b = (beta - mean * gamma * invstd) * 127.5 / MaxAbs(calib range),
 * out = saturate(nearest-even((w / sqrt(1 + eps)) * x + b)), with max(0, .) before the
 * rounding for the relu form; the output range is (min_calib, max_calib), which the
 * operator requires.  The factor and offset follow the reference's own file; the
 * normalisation itself (the second division by sqrt(1 + eps), the order of multiply and
 * add, the rounding) runs inside oneDNN there and is not pinned by its sources (its test
 * accepts rtol 0.1, atol 8).  workspace: mxq_quantized_batch_norm_workspace(channels)
 * bytes, 4-byte aligned. */
size_t mxq_quantized_batch_norm_workspace(int64_t channels);
int mxq_quantized_batch_norm(void* stream, const void* data, int data_type, const float* gamma,
                             const float* beta, const float* moving_mean,
                             const float* moving_var, const float* min_data,
                             const float* max_data, int8_t* out, float* omin, float* omax,
                             int64_t outer, int64_t channels, int64_t inner, double eps,
                             float min_calib, float max_calib, int relu, void* workspace,
                             size_t workspace_bytes);

/* ---- _contrib_quantized_concat -----------------------------------------------------
 * Replaces DNNLQuantizedConcatForward
 * (src/operator/quantization/dnnl/dnnl_quantized_concat.cc:41-115; cpu-only in the
 * reference).  Input i is [outer, in_axis[i], inner] contiguous, the output
 * [outer, sum in_axis, inner].  Output range = hull of the input ranges and 0; out_type is
 * int8 as soon as one input is (quantized_concat.cc:83-103).  An input whose scale equals
 * the output's is copied, any other is rescaled: saturate(nearest-even(x * out_scale /
 * in_scale)) in binary32 (oneDNN's reorder; same caveat as above).  in, in_type, in_min,
 * in_max, in_axis are host arrays of num_args entries; the data and range pointers in
 * them are device pointers. */
int mxq_quantized_concat(void* stream, int num_args, const void* const* in, const int* in_type,
                         const float* const* in_min, const float* const* in_max,
                         const int64_t* in_axis, int64_t outer, int64_t inner, void* out,
                         int out_type, float* omin, float* omax);

/* ---- _contrib_quantized_fully_connected ----------------------------------
 * Replaces QuantizedFullyConnectedForwardGPU
 * (src/operator/quantization/quantized_fully_connected.cu:58-138): cublasGemmEx
 * (s8 x s8 -> s32, data [M,K] row-major, weight [N,K] row-major), the
 * QuantizationRangeForS8S8MultiplicationStruct launch and QuantizedBiasAddKernel.
 * The bias is added exactly, as the CPU operator does
 * (quantized_fully_connected.cc:149-174: the int8 bias is rescaled to int32 once
 * and summed in integers), not through the GPU kernel's float round trip.
 *   bias        int8 [N] or NULL (then min_bias/max_bias are ignored)
 *   out32       int32 [M,N] or NULL
 *   omin, omax  output range (always written)
 *   out8        int8 [M,N] or NULL: fused _contrib_requantize of the
 *               accumulator with the calibrated range (min_calib, max_calib),
 *               bit-identical to mxq_requantize on out32; relu != 0 clamps the
 *               int8 at zero; rmin/rmax receive the requantized range.
 * At least one of out32 / out8 must be given.
 *   workspace   device scratch (16-byte aligned) or NULL.  Shapes with few output tiles and
 *               a long K are split along K over several work-groups per tile, which leave
 *               their int32 partial sums in the workspace (integer addition is
 *               associative: the result is the unsplit one bit for bit); this is the
 *               operator's kTempSpace (quantized_fully_connected.cc:369-372).
 *               mxq_quantized_fc_workspace() returns the bytes with which the call takes
 *               its fastest route (0 when it would not split; fused_int8_only != 0 says
 *               that only out8 will be given); with less, or NULL, nothing is split. */
size_t mxq_quantized_fc_workspace(int M, int N, int K, int fused_int8_only);
int mxq_quantized_fc(void* stream, const int8_t* data, const int8_t* weight, const int8_t* bias,
                     int M, int N, int K, const float* min_data, const float* max_data,
                     const float* min_weight, const float* max_weight, const float* min_bias,
                     const float* max_bias, int32_t* out32, float* omin, float* omax,
                     int8_t* out8, float* rmin, float* rmax, int relu, float min_calib,
                     float max_calib, void* workspace, size_t workspace_bytes);

/* _contrib_quantized_fully_connected -> _contrib_requantize -> _contrib_dequantize in one
 * launch: the three operators a quantized graph runs where a float consumer follows the
 * layer (quantized_fully_connected.cu:58-138, requantize-inl.h:89-125 with a calibrated
 * range, dequantize-inl.h:64-75).  out_f32 [M,N] receives float(q) * (R / 127) with q the
 * requantized int8 value and R = max(|min_calib|, |max_calib|): bit-identical to
 * mxq_dequantize(mxq_requantize(out32)) element by element; relu != 0 clamps q at zero
 * first.  omin/omax and rmin/rmax are written as by mxq_quantized_fc.  The int8 tensor
 * between the operators is never stored.  Workspace as for mxq_quantized_fc (size it with
 * fused_int8_only = 0). */
int mxq_quantized_fc_f32(void* stream, const int8_t* data, const int8_t* weight,
                         const int8_t* bias, int M, int N, int K, const float* min_data,
                         const float* max_data, const float* min_weight, const float* max_weight,
                         const float* min_bias, const float* max_bias, float* out_f32,
                         float* omin, float* omax, float* rmin, float* rmax, int relu,
                         float min_calib, float max_calib, void* workspace,
                         size_t workspace_bytes);

/* _contrib_quantized_fully_connected -> _contrib_requantize -> _contrib_quantized_elemwise_add
 * (-> _contrib_quantized_act) in one launch: a layer whose requantized int8 output is added
 * to a second int8 tensor of the same shape, the residual sum of a bottleneck block
 * (quantized_fully_connected.cu:58-138, requantize-inl.h:89-125,
 * quantized_elemwise_add.cc:30-134 / dnnl/dnnl_quantized_elemwise_add.cc:134-257 with a
 * calibrated int8 output, quantized_activation.cc:84-120).  In NHWC a 1x1 unit-stride
 * unpadded convolution is this call on the flattened pixels (M = N*H*W, K = C, N = O).
 *   residual       int8 [M,N], range (min_residual, max_residual)
 *   min/max_calib  the layer's own requantization range, as for mxq_quantized_fc
 *   sum_*_calib    the sum's calibrated range; rmin / rmax receive it
 *   sum_relu != 0  clamps the sum at zero
 * out8 is bit-identical to mxq_quantized_elemwise_add(out8 of mxq_quantized_fc, residual)
 * followed by mxq_quantized_relu; neither intermediate tensor is stored.  (The element
 * rounding of the sum is this library's own choice: in the reference it happens inside
 * oneDNN and its parity is unpinned, as for mxq_quantized_elemwise_add.)  out8 may be the
 * residual's own buffer (the shortcut updated in place).  Workspace as for
 * mxq_quantized_fc with fused_int8_only = 1. */
int mxq_quantized_fc_sum(void* stream, const int8_t* data, const int8_t* weight,
                         const int8_t* bias, int M, int N, int K, const float* min_data,
                         const float* max_data, const float* min_weight, const float* max_weight,
                         const float* min_bias, const float* max_bias, const int8_t* residual,
                         const float* min_residual, const float* max_residual, int8_t* out8,
                         float* omin, float* omax, float* rmin, float* rmax, float min_calib,
                         float max_calib, float sum_min_calib, float sum_max_calib, int sum_relu,
                         void* workspace, size_t workspace_bytes);

/* mxq_quantized_fc_sum for a sum that is calibrated behind the operator: the layer's
 * requantized int8 output and the residual are added in int32 over the sum's own range
 * (_contrib_quantized_elemwise_add without a calibrated range) and that sum is requantized
 * over (sum_min_calib, sum_max_calib) (_contrib_requantize), which is the graph QuantizeGraph
 * makes of an elemwise_add between two layers; sum_relu != 0 clamps at zero.  out8 is
 * bit-identical to the operators one after the other; rmin / rmax receive the requantized
 * range.
 * `pairs` is null, or what mxq_sum_requant_pairs left on the device for these very ranges. */
int mxq_quantized_fc_sum_requant(void* stream, const int8_t* data, const int8_t* weight,
                                 const int8_t* bias, int M, int N, int K, const float* min_data,
                                 const float* max_data, const float* min_weight,
                                 const float* max_weight, const float* min_bias,
                                 const float* max_bias, const int8_t* residual,
                                 const float* min_residual, const float* max_residual,
                                 int8_t* out8, float* omin, float* omax, float* rmin, float* rmax,
                                 float min_calib, float max_calib, float sum_min_calib,
                                 float sum_max_calib, int sum_relu, const void* pairs,
                                 void* workspace, size_t workspace_bytes);

/* The layers above, and mxq_quantized_conv_nhwc, for ranges that stay: mxq_prepare_layer computes
 * what a launch derives from the six ranges, the calibrated range and the bias once, into
 * 64 + 4 * N bytes on the device (16-byte aligned); the _prepared entries take it instead of them,
 * write the same int8 (or dequantized float) output and no ranges. */
int mxq_prepare_layer(void* stream, const int8_t* bias, int N, const float* min_data,
                      const float* max_data, const float* min_weight, const float* max_weight,
                      const float* min_bias, const float* max_bias, float min_calib,
                      float max_calib, void* prepared);
/* Looks for short forms of the layer's requantize that give the same int8 for every accumulator and
 * notes them in what mxq_prepare_layer wrote, for the launches that use them. */
int mxq_prepare_forms(void* stream, void* prepared);
int mxq_quantized_fc_prepared(void* stream, const int8_t* data, const int8_t* weight,
                              const void* prepared, int M, int N, int K, int8_t* out8,
                              float* out_f32, int relu, float min_calib, float max_calib,
                              void* workspace, size_t workspace_bytes);
int mxq_quantized_fc_sum_prepared(void* stream, const int8_t* data, const int8_t* weight,
                                  const void* prepared, int M, int N, int K,
                                  const int8_t* residual, const float* min_residual,
                                  const float* max_residual, int8_t* out8, float min_calib,
                                  float max_calib, float sum_min_calib, float sum_max_calib,
                                  int sum_relu, int requant, const void* pairs, void* workspace,
                                  size_t workspace_bytes);
int mxq_quantized_conv_nhwc_prepared(void* stream, const int8_t* data, const int8_t* weight,
                                     const void* prepared, int N, int H, int W, int C, int O,
                                     int KH, int KW, int stride_h, int stride_w, int pad_h,
                                     int pad_w, int dilate_h, int dilate_w, int8_t* out8, int relu,
                                     float min_calib, float max_calib, void* workspace,
                                     size_t workspace_bytes);

/* Two 1 x 1 convolutions of the same images, both prepared, in one launch (two where the operands
 * are unaligned or _fits is 0). */
int mxq_quantized_conv_pair_fits(int N, int H, int W, int C, int O1, int O2, int stride_h,
                                 int stride_w);
int mxq_quantized_conv_pair_prepared(void* stream, const int8_t* data, int N, int H, int W, int C,
                                     int stride_h, int stride_w, const int8_t* weight1,
                                     const void* prepared1, int O1, int8_t* out1, int relu1,
                                     float min_calib1, float max_calib1, const int8_t* weight2,
                                     const void* prepared2, int O2, int8_t* out2, int relu2,
                                     float min_calib2, float max_calib2);

/* A 3 x 3 convolution of stride 1 and padding 1, prepared, over 256 channels and more (a multiple),
 * with its weights [O][3][3][C] laid out beforehand. */
int mxq_quantized_conv3x3_fits(int N, int H, int W, int C, int O);
size_t mxq_quantized_conv3x3_weights(int C, int O);
int mxq_pack_conv3x3_weights(void* stream, const int8_t* in, int C, int O, int8_t* out);
int mxq_quantized_conv3x3(void* stream, const int8_t* data, const int8_t* weights,
                          const void* prepared, int N, int H, int W, int C, int O, int8_t* out8,
                          int relu);

/* A stem: a 4 x 4 convolution of stride 1 over 16 channels, prepared, and the 3 x 3 maximum of
 * stride 2 and padding 1 behind it in one launch; out8 is [N][pooled_h][pooled_w][O]. */
int mxq_quantized_conv_pool_fits(int N, int H, int W, int C, int O, int KH, int KW, int pad_h,
                                 int pad_w, int pooled_h, int pooled_w);
int mxq_quantized_conv_pool(void* stream, const int8_t* data, const int8_t* weight,
                            const void* prepared, int N, int H, int W, int C, int O, int KH,
                            int KW, int pad_h, int pad_w, int pooled_h, int pooled_w, int8_t* out8,
                            int relu);

/* Looks for a short form of that sum with sum_relu != 0 over ranges that stay: two products and
 * one rounding that give the same int8 for every pair of int8 operands, which is tried out on
 * the device.  Writes 12 bytes to `pairs` (device, 4-byte aligned), among them whether one was
 * found; the fused launch takes it from there, without it the result is the same. */
int mxq_sum_requant_pairs(void* stream, float min_calib, float max_calib,
                          float min_residual, float max_residual, float sum_min_calib,
                          float sum_max_calib, void* pairs);

/* ---- _contrib_quantized_conv ----------------------------------------------
 * Replaces QuantizedCuDNNConvOp::Forward
 * (src/operator/quantization/quantized_conv.cu:101-219): the NHWC int8
 * cudnnConvolutionForward, the float->int32 cast, the range kernel and the bias
 * kernel.  Operands are NHWC here (data [N,H,W,C], weight [O,KH,KW,C], output
 * [N,OH,OW,O]); the layout adapters below replace the three TransposeImpl calls
 * (:147-148,183) for callers holding the operator's NCHW tensors.  Epilogue
 * and workspace arguments as for mxq_quantized_fc (the reference passes cuDNN its own
 * workspace out of the operator's temp space, quantized_conv.cu:121-177). */
size_t mxq_quantized_conv_workspace(int N, int H, int W, int C, int O, int KH, int KW,
                                    int stride_h, int stride_w, int pad_h, int pad_w,
                                    int dilate_h, int dilate_w, int fused_int8_only);
int mxq_quantized_conv_nhwc(void* stream, const int8_t* data, const int8_t* weight,
                            const int8_t* bias, int N, int H, int W, int C, int O, int KH,
                            int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                            int dilate_h, int dilate_w, const float* min_data,
                            const float* max_data, const float* min_weight,
                            const float* max_weight, const float* min_bias,
                            const float* max_bias, int32_t* out32, float* omin, float* omax,
                            int8_t* out8, float* rmin, float* rmax, int relu, float min_calib,
                            float max_calib, void* workspace, size_t workspace_bytes);
/* The same convolution with the int32 output written as the operator's own layout,
 * [N,O,OH,OW]: the kernel's epilogue stores channel planes directly, which replaces the
 * third TransposeImpl (quantized_conv.cu:183) and the NHWC int32 buffer it reads. */
int mxq_quantized_conv_nhwc_out_nchw(void* stream, const int8_t* data, const int8_t* weight,
                                     const int8_t* bias, int N, int H, int W, int C, int O,
                                     int KH, int KW, int stride_h, int stride_w, int pad_h,
                                     int pad_w, int dilate_h, int dilate_w,
                                     const float* min_data, const float* max_data,
                                     const float* min_weight, const float* max_weight,
                                     const float* min_bias, const float* max_bias,
                                     int32_t* out32_nchw, float* omin, float* omax,
                                     void* workspace, size_t workspace_bytes);

/* _contrib_quantized_conv on the operator's own tensors: data int8 [N,C,H,W], weight int8
 * [O,C,KH,KW], bias int8 [O] or NULL, out32 int32 [N,O,OH,OW] -- everything
 * QuantizedCuDNNConvOp::Forward does between its inputs and its outputs
 * (src/operator/quantization/quantized_conv.cu:101-219, layout rule quantized_conv.cc:38-45),
 * the three TransposeImpl calls included (:145-148,183).  Unpadded 1 x 1 convolutions over
 * 16 | C channels never leave the channel-plane layout (strided ones and planes that are
 * no multiple of 16 bytes through a gathering loader in the same kernel or, where that
 * would fetch single bytes, after the pixels they read were gathered into the workspace);
 * every other geometry goes through the layout adapters and
 * mxq_quantized_conv_nhwc_out_nchw inside this call.
 * `workspace` (16-byte aligned) must hold mxq_quantized_conv_nchw_workspace() bytes: the
 * operator's kTempSpace (quantized_conv.cu:121-160 asks for three tensor copies plus
 * cuDNN's workspace there; 0 here for most unpadded 1 x 1 layers).  operands_aligned16 != 0
 * says that data and weight both start on 16-byte marks, as a framework's allocations do;
 * with 0 the query returns enough for the adapter route as well, which every geometry and
 * alignment can take. */
size_t mxq_quantized_conv_nchw_workspace(int N, int C, int H, int W, int O, int KH, int KW,
                                         int stride_h, int stride_w, int pad_h, int pad_w,
                                         int dilate_h, int dilate_w, int operands_aligned16);
int mxq_quantized_conv_nchw(void* stream, const int8_t* data, const int8_t* weight,
                            const int8_t* bias, int N, int C, int H, int W, int O, int KH, int KW,
                            int stride_h, int stride_w, int pad_h, int pad_w, int dilate_h,
                            int dilate_w, const float* min_data, const float* max_data,
                            const float* min_weight, const float* max_weight,
                            const float* min_bias, const float* max_bias, int32_t* out32,
                            float* omin, float* omax, void* workspace, size_t workspace_bytes);

/* ---- networks held as NHWC ---------------------------------------------------
 * For a caller that keeps int8 activations as [N,H,W,C_padded] between the layers, C_padded
 * the channel count rounded up to 16 and the channels past C zero (zero weights and a zero
 * bias keep them zero through every layer).
 * mxq_quantize_to_nhwc: calibrated quantize_v2 (int8) of a float NCHW image straight into that
 * layout; space_to_depth != 0 into the layout of mxq_nchw_to_s2d_nhwc_i8.
 * mxq_quantize_to_s2d: that, with H2 and W2 given; each may be one more than that layout's, the
 * last row or column then holds zeros alone.
 * mxq_quantized_pooling_nhwc: mxq_quantized_pooling_nchw's windows and rounding on int8 of that
 * layout (C a multiple of 16); the range passes through and is left to the caller.
 * mxq_pack_weight: OIHW int8 -> [O_padded,KH,KW,C_padded] with zeros, or the weight of the
 * space-to-depth form ([O_padded,(KH+1)/2,(KW+1)/2,C_padded]).
 * mxq_nhwc_pad_to_nchw_i8: back to [N,C,H,W]. */
int mxq_quantize_to_nhwc(void* stream, const float* in, int8_t* out, float* omin, float* omax,
                         int N, int C, int H, int W, int C_padded, int space_to_depth, int off_h,
                         int off_w, float min_calib, float max_calib);
int mxq_quantize_to_s2d(void* stream, const float* in, int8_t* out, float* omin, float* omax,
                        int N, int C, int H, int W, int C_padded, int off_h, int off_w, int H2,
                        int W2, float min_calib, float max_calib);
int mxq_quantized_pooling_nhwc(void* stream, const int8_t* in, int N, int H, int W, int C,
                               int kernel_h, int kernel_w, int stride_h, int stride_w, int pad_h,
                               int pad_w, int OH, int OW, int pool_type, int count_include_pad,
                               int8_t* out);
int mxq_pack_weight(void* stream, const int8_t* in, int8_t* out, int O, int C, int KH, int KW,
                    int O_padded, int C_padded, int space_to_depth);
int mxq_nhwc_pad_to_nchw_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int C_padded);

/* The tail of a residual block over NHWC activations as one launch (channel counts multiples of
 * 16, ranges that stay): 3 x 3 convolution (stride and pad 1) C -> C_mid, requantize, relu if
 * relu_first; 1 x 1 convolution C_mid -> C_out and the sum with `residual` as
 * mxq_quantized_fc_sum_prepared with requant and sum_relu computes it, into `out`; and, unless
 * C_next is 0, the 1 x 1 convolution C_out -> C_next that reads that sum, requantize, relu if
 * relu_third, into `next`.  All three layers' int8 results are those of the launches one by one;
 * the two that only this launch reads are not stored.
 * mxq_quantized_block_fits: whether a block of this shape can run that way and is faster for it.
 * mxq_pack_block_weights: the layers' NHWC weights [C_mid,3,3,C], [C_out,C_mid], [C_next,C_out]
 * into the mxq_quantized_block_weights() bytes that the launch reads (16-byte aligned).
 * mxq_prepare_block: from what mxq_prepare_layer made of the layers (their scales; the launch
 * takes their bias from there), the residual's range and the calibrated ranges of the second
 * layer and of the sum, the mxq_quantized_block_forms() bytes that the launch reads (16-byte
 * aligned). */
int mxq_quantized_block_fits(int N, int H, int W, int C, int C_mid, int C_out, int C_next);
size_t mxq_quantized_block_weights(int C, int C_mid, int C_out, int C_next);
int mxq_pack_block_weights(void* stream, const int8_t* first, const int8_t* second,
                           const int8_t* third, int C, int C_mid, int C_out, int C_next,
                           int8_t* out);
size_t mxq_quantized_block_forms(void);
int mxq_prepare_block(void* stream, const void* prepared_first, const void* prepared_second,
                      const void* prepared_third, const float* min_residual,
                      const float* max_residual, float min_calib, float max_calib,
                      float sum_min_calib, float sum_max_calib, void* forms);
int mxq_quantized_block(void* stream, const int8_t* data, const int8_t* weights,
                        const void* forms, const void* prepared_first,
                        const void* prepared_second, const void* prepared_third, int N, int H,
                        int W, int C, int C_mid, int C_out, int C_next, const int8_t* residual,
                        int8_t* out, int8_t* next, int relu_first, int relu_third);

/* ---- calibration -----------------------------------------------------------
 * What the calibration collectors take of a float tensor
 * (python/mxnet/contrib/quantization.py:269-361, numpy on the host in the reference).
 * mxq_minmax_f32: smallest and largest value into two device floats, both NaN if there is a
 * NaN; workspace as for mxq_quantize_v2.
 * mxq_histogram_f32: counts[k] of the values with edges[k] <= x < edges[k + 1] (the last bin
 * includes its upper edge), `bins` + 1 increasing edges and `bins` counts on the device;
 * values outside and NaN are not counted; n < 2^32.
 * mxq_symmetric_histogram_f32: both in one go, without a word from the host between them.  `out`, on
 * the device, receives the two extreme values, 1 or 0, and the `bins` counts (of at most 2^24) over
 * [-th, th], its edges as numpy.histogram computes them in float32; th of NaN: the larger magnitude
 * of the two.  0 where those edges do not increase or th is not finite: nothing is counted then.  The
 * workspace is 16-byte aligned.
 * mxq_symmetric_histogram_inside_f32: the same, but 0 as well where a value lies beyond th. */
size_t mxq_minmax_f32_workspace(size_t n);
int mxq_minmax_f32(void* stream, const float* in, size_t n, float* out_min, float* out_max,
                   void* workspace, size_t workspace_bytes);
int mxq_histogram_f32(void* stream, const float* in, size_t n, const float* edges, int bins,
                      uint32_t* counts);
size_t mxq_symmetric_histogram_f32_workspace(size_t n, int bins);
int mxq_symmetric_histogram_f32(void* stream, const float* in, size_t n, int bins, float th,
                                uint32_t* out, void* workspace, size_t workspace_bytes);
int mxq_symmetric_histogram_inside_f32(void* stream, const float* in, size_t n, int bins, float th,
                                       uint32_t* out, void* workspace, size_t workspace_bytes);

/* Entropy calibration: bounds [lower, upper] of what mxq_calibrate_entropy's float sums give for
 * every candidate threshold, narrowest first, of up to 16 histograms (`hist`, on the device, one
 * behind the other, finite, none negative, less than 2^31 counts each; `bins` odd, up to 32767, and
 * `levels` of 3 and more, on the host), as doubles on the device; (-inf, inf) where none are known,
 * (inf, inf) for a candidate without a quantized distribution. */
size_t mxq_entropy_bounds_workspace(int count, const int* bins, const int* levels);
int mxq_entropy_bounds(void* stream, int count, const float* hist, const int* bins,
                       const int* levels, double* bounds, void* workspace,
                       size_t workspace_bytes);

/* [N,C,H,W] int8 -> [N,H,W,C] int8 (also OIHW -> OHWI for the weight). */
int mxq_nchw_to_nhwc_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H, int W);
/* The same with the channel extent of the output padded to C_padded >= C with zeros
 * ([N,H,W,C_padded]): zero channels add nothing to a convolution, and a channel count
 * that is a multiple of 16 takes mxq_quantized_conv_nhwc's fast path. */
int mxq_nchw_to_nhwc_pad_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int C_padded);
/* Space-to-depth by 2 on the way: [N,C,H,W] -> [N,H2,W2,C_padded] with
 * out[n][h2][w2][(dh*2+dw)*C + c] = in[n][c][2*h2 - off_h + dh][2*w2 - off_w + dw] (zero
 * outside the image; channels 4*C..C_padded-1 zero), H2 = (H + off_h + 1) / 2, likewise W2,
 * off in {0,1}.  A KxK stride-2 convolution with padding p over C channels equals the
 * ceil(K/2) x ceil(K/2) unit-stride convolution with padding (p - off) / 2 over this tensor
 * (off = p mod 2) and the weight transformed the same way with off = 0, whenever both
 * give the same output extent; few-channel stride-2 stems run that way. */
int mxq_nchw_to_s2d_nhwc_i8(void* stream, const int8_t* in, int8_t* out, int N, int C, int H,
                            int W, int off_h, int off_w, int C_padded);
/* [N,H,W,C] -> [N,C,H,W]; elem_bytes 1 (int8) or 4 (int32). */
int mxq_nhwc_to_nchw(void* stream, const void* in, void* out, int N, int C, int H, int W,
                     int elem_bytes);

#ifdef __cplusplus
}
#endif
#endif /* MXQ_H_ */
