"""ctypes binding of libmxq_hip.so.  There is no fallback: if the library is
missing or a symbol is absent the import raises."""
import ctypes
import os

# before the library below: the HIP runtime torch brings has to be the process's only one
import torch  # noqa: F401

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmxq_hip.so")

# element type codes = mshadow::TypeFlag
FLOAT32, UINT8, INT32, INT8 = 0, 3, 4, 5


class MXQError(RuntimeError):
    """A C-ABI call returned non-zero; carries mxq_last_error()."""


if not os.path.exists(LIB_PATH):
    raise ImportError(
        "libmxq_hip.so is not built: run `python -c 'import __graft_entry__ as g; g.build()'` "
        "(or python mxnet_amd/build.py) first; there is no CPU fallback")

lib = ctypes.CDLL(LIB_PATH)

_p = ctypes.c_void_p
_sz = ctypes.c_size_t
_i = ctypes.c_int
_f = ctypes.c_float

# every symbol include/mxq.h declares, with its signature
SIGNATURES = {
    "mxq_last_error": (ctypes.c_char_p, []),
    "mxq_abi_version": (_i, []),
    "mxq_quantize_v2_workspace": (_sz, [_sz]),
    "mxq_quantize_v2": (_i, [_p, _p, _p, _p, _p, _sz, _i, _i, _f, _f, _p, _sz]),
    "mxq_quantize_v2_noalloc": (_i, [_p, _p, _p, _p, _p, _sz, _i, _i, _f, _f]),
    "mxq_quantize": (_i, [_p, _p, _p, _p, _p, _p, _p, _sz, _i]),
    "mxq_quantize_v2_passthrough": (_i, [_p, _p, _p, _p, _p, _sz, _i, _i, _f, _f]),
    "mxq_requantize_workspace": (_sz, [_sz]),
    "mxq_requantize": (_i, [_p, _p, _p, _p, _p, _p, _p, _sz, _i, _f, _f, _p, _sz]),
    "mxq_dequantize": (_i, [_p, _p, _i, _p, _p, _p, _sz]),
    "mxq_quantized_relu": (_i, [_p, _p, _p, _p, _p, _p, _p, _sz]),
    "mxq_quantized_pooling_nchw": (_i, [_p, _p, _i] + [_i] * 12 + [_i, _i, _p, _p, _p, _p, _p]),
    "mxq_quantized_flatten": (_i, [_p, _p, _p, _p, _p, _p, _p, _sz]),
    "mxq_quantized_elemwise_add": (_i, [_p, _p, _i, _p, _i, _p, _p, _p, _p, _p, _i, _p, _p, _sz,
                                        _i, _f, _f]),
    "mxq_quantized_broadcast_add": (_i, [_p, _p, _i, _i, _p, _p, _i, _i, _p, _p, _p, _p, _p, _p,
                                         _i, _p, _p, _i, _f, _f]),
    "mxq_quantized_elemwise_mul": (_i, [_p, _p, _p, _p, _p, _p, _p, _p, _i, _p, _p, _sz, _i, _f,
                                        _f]),
    "mxq_quantized_embedding": (_i, [_p, _p, _i, _p, _p, _p, _p, _p, _p, _sz, ctypes.c_int64,
                                     ctypes.c_int64]),
    "mxq_quantized_transpose": (_i, [_p, _p, _p, _p, _p, _p, _p, _i, _p, _p]),
    "mxq_quantize_asym_workspace": (_sz, [_sz]),
    "mxq_quantize_asym": (_i, [_p, _p, _i, _p, _p, _p, _sz, _i, _f, _f, _p, _sz]),
    "mxq_quantized_batch_norm_workspace": (_sz, [ctypes.c_int64]),
    "mxq_quantized_batch_norm": (_i, [_p, _p, _i] + [_p] * 6 + [_p, _p, _p] +
                                 [ctypes.c_int64] * 3 + [ctypes.c_double, _f, _f, _i, _p, _sz]),
    "mxq_quantized_concat": (_i, [_p, _i, _p, _p, _p, _p, _p, ctypes.c_int64, ctypes.c_int64, _p,
                                  _i, _p, _p]),
    "mxq_quantized_fc_workspace": (_sz, [_i, _i, _i, _i]),
    "mxq_quantized_fc": (_i, [_p, _p, _p, _p, _i, _i, _i] + [_p] * 6 + [_p, _p, _p, _p, _p, _p,
                              _i, _f, _f, _p, _sz]),
    "mxq_quantized_fc_f32": (_i, [_p, _p, _p, _p, _i, _i, _i] + [_p] * 6 + [_p, _p, _p, _p, _p,
                                  _i, _f, _f, _p, _sz]),
    "mxq_quantized_fc_sum": (_i, [_p, _p, _p, _p, _i, _i, _i] + [_p] * 6 + [_p, _p, _p] +
                             [_p, _p, _p, _p, _p, _f, _f, _f, _f, _i, _p, _sz]),
    "mxq_quantized_fc_sum_requant": (_i, [_p, _p, _p, _p, _i, _i, _i] + [_p] * 6 + [_p, _p, _p] +
                                     [_p, _p, _p, _p, _p, _f, _f, _f, _f, _i, _p, _p, _sz]),
    "mxq_prepare_layer": (_i, [_p, _p, _i] + [_p] * 6 + [_f, _f, _p]),
    "mxq_quantized_fc_prepared": (_i, [_p] * 4 + [_i] * 3 + [_p, _p, _i, _f, _f, _p, _sz]),
    "mxq_quantized_fc_sum_prepared": (_i, [_p] * 4 + [_i] * 3 + [_p] * 4 + [_f] * 4 +
                                      [_i, _i, _p, _p, _sz]),
    "mxq_prepare_forms": (_i, [_p, _p]),
    "mxq_quantized_conv3x3_fits": (_i, [_i] * 5),
    "mxq_quantized_conv3x3_weights": (_sz, [_i] * 2),
    "mxq_pack_conv3x3_weights": (_i, [_p, _p, _i, _i, _p]),
    "mxq_quantized_conv3x3": (_i, [_p] * 4 + [_i] * 5 + [_p, _i]),
    "mxq_quantized_conv_pool_fits": (_i, [_i] * 11),
    "mxq_quantized_conv_pool": (_i, [_p] * 4 + [_i] * 11 + [_p, _i]),
    "mxq_quantized_conv_pair_fits": (_i, [_i] * 8),
    "mxq_quantized_conv_pair_prepared": (_i, [_p] * 2 + [_i] * 6 +
                                         [_p, _p, _i, _p, _i, _f, _f] * 2),
    "mxq_quantized_conv_nhwc_prepared": (_i, [_p] * 4 + [_i] * 13 +
                                         [_p, _i, _f, _f, _p, _sz]),
    "mxq_sum_requant_pairs": (_i, [_p, _f, _f, _f, _f, _f, _f, _p]),
    "mxq_quantized_conv_workspace": (_sz, [_i] * 14),
    "mxq_quantized_conv_nhwc": (_i, [_p, _p, _p, _p] + [_i] * 13 + [_p] * 6 +
                                [_p, _p, _p, _p, _p, _p, _i, _f, _f, _p, _sz]),
    "mxq_quantized_conv_nhwc_out_nchw": (_i, [_p, _p, _p, _p] + [_i] * 13 + [_p] * 6 +
                                         [_p, _p, _p, _p, _sz]),
    "mxq_quantized_conv_nchw_workspace": (_sz, [_i] * 14),
    "mxq_quantized_conv_nchw": (_i, [_p, _p, _p, _p] + [_i] * 13 + [_p] * 6 +
                                [_p, _p, _p, _p, _sz]),
    "mxq_quantize_to_nhwc": (_i, [_p] * 5 + [_i] * 8 + [_f, _f]),
    "mxq_quantize_to_s2d": (_i, [_p] * 5 + [_i] * 9 + [_f, _f]),
    "mxq_quantized_pooling_nhwc": (_i, [_p, _p] + [_i] * 14 + [_p]),
    "mxq_pack_weight": (_i, [_p, _p, _p] + [_i] * 7),
    "mxq_quantized_block_fits": (_i, [_i] * 7),
    "mxq_quantized_block_weights": (_sz, [_i] * 4),
    "mxq_pack_block_weights": (_i, [_p] * 4 + [_i] * 4 + [_p]),
    "mxq_quantized_block_forms": (_sz, []),
    "mxq_prepare_block": (_i, [_p] * 6 + [_f] * 4 + [_p]),
    "mxq_quantized_block": (_i, [_p] * 7 + [_i] * 7 + [_p] * 3 + [_i, _i]),
    "mxq_nhwc_pad_to_nchw_i8": (_i, [_p, _p, _p] + [_i] * 5),
    "mxq_minmax_f32_workspace": (_sz, [_sz]),
    "mxq_minmax_f32": (_i, [_p, _p, _sz, _p, _p, _p, _sz]),
    "mxq_histogram_f32": (_i, [_p, _p, _sz, _p, _i, _p]),
    "mxq_symmetric_histogram_f32_workspace": (_sz, [_sz, _i]),
    "mxq_symmetric_histogram_f32": (_i, [_p, _p, _sz, _i, _f, _p, _p, _sz]),
    "mxq_symmetric_histogram_inside_f32": (_i, [_p, _p, _sz, _i, _f, _p, _p, _sz]),
    "mxq_entropy_bounds_workspace": (_sz, [_i, ctypes.POINTER(_i), ctypes.POINTER(_i)]),
    "mxq_entropy_bounds": (_i, [_p, _i, _p, ctypes.POINTER(_i), ctypes.POINTER(_i), _p, _p, _sz]),
    "mxq_nchw_to_nhwc_i8": (_i, [_p, _p, _p, _i, _i, _i, _i]),
    "mxq_nchw_to_nhwc_pad_i8": (_i, [_p, _p, _p, _i, _i, _i, _i, _i]),
    "mxq_nchw_to_s2d_nhwc_i8": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _i]),
    "mxq_nhwc_to_nchw": (_i, [_p, _p, _p, _i, _i, _i, _i, _i]),
}

for _name, (_res, _args) in SIGNATURES.items():
    _fn = getattr(lib, _name)  # AttributeError if the library lacks the symbol
    _fn.restype = _res
    _fn.argtypes = _args

# test-only twins of the FC and convolution entry points (tests/mxq_test_hooks.h, not part
# of include/mxq.h): the same arguments followed by the tile configuration, the split-K
# factor and, for the FC, the streaming kernel's work-groups per CU (0 = choose); what a block's
# launch reads of LDS; what is chosen for a layer; and the functions that the entropy bounds are made of
TEST_HOOKS = {
    "mxq_test_quantized_fc": (_i, SIGNATURES["mxq_quantized_fc"][1] + [_i, _i, _i]),
    "mxq_test_quantized_fc_sum": (_i, SIGNATURES["mxq_quantized_fc_sum"][1] + [_i, _i, _i]),
    "mxq_test_quantized_fc_sum_requant": (_i, SIGNATURES["mxq_quantized_fc_sum_requant"][1] +
                                          [_i, _i, _i]),
    "mxq_test_quantized_fc_f32": (_i, SIGNATURES["mxq_quantized_fc_f32"][1] + [_i, _i]),
    "mxq_test_quantized_conv_nhwc": (_i, SIGNATURES["mxq_quantized_conv_nhwc"][1] + [_i, _i]),
    "mxq_test_quantized_conv_nchw": (_i, SIGNATURES["mxq_quantized_conv_nchw"][1] + [_i]),
    "mxq_test_block_lds": (_i, [_i] * 8 + [ctypes.POINTER(_i)] * 2),
    "mxq_test_fc_plan": (_i, [_i] * 6 + [_p, _sz] + [ctypes.POINTER(_i)] * 2),
    "mxq_test_conv_plan": (_i, [_i] * 13 + [_p, _sz] + [ctypes.POINTER(_i)] * 2),
    "mxq_test_entropy_functions": (_i, [_p, _p, _p, _sz, _p, _p, _p]),
}
for _name, (_res, _args) in TEST_HOOKS.items():
    _fn = getattr(lib, _name)
    _fn.restype = _res
    _fn.argtypes = _args


def last_error():
    return lib.mxq_last_error().decode()


def check(rc):
    if rc != 0:
        raise MXQError(last_error())
