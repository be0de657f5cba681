// The kernel for contractions with few output tiles (mxq_few_tiles.hip): its arguments, its
// launchers and the rule that chooses it.
#ifndef MXQ_FEW_TILES_H_
#define MXQ_FEW_TILES_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "mxq_gemm.h"

namespace mxq {

struct FewTilesArgs {
  const int8_t* data;    // [M][K], or NHWC images of a convolution
  const int8_t* weight;  // [N][K]
  int M, N, K;
  int ldo;               // output row pitch in elements
  Epilogue epi;
  // convolution only
  int images, H, W, C, KW, sh, sw, ph, pw, dh, dw, OH, OW;
  uint32_t magic_c, magic_kw;  // filled by the launcher
};

inline long few_tiles_count(long M, long N) { return ((M + 31) / 32) * ((N + 31) / 32); }

// Where the kernel is chosen for aligned operands: no more 32 x 32 tiles than CUs, so that the
// 64 x 64 tiles of the other kernels would leave most of the chip idle (196 x 1024 -> 1024, 224
// tiles: 4.1 us against 5.2; 784 x 1024 -> 512, 400 tiles: 5.7 against 5.2), and a reduction of
// at least two blocks (at 64 bytes the tiled kernels are level or ahead).  From 8192 on
// the tiled kernels split the reduction over work-groups and keep all but the smallest outputs, from 32768 on
// these too where the caller brought room for it (us, here and there: 121 x 34800 -> 153 23.2 / 17.5, 48 x
// 33200 -> 686 23.5 / 18.2, 192 x 25088 -> 81 16.2 / 15.4, but 512 x 17248 -> 106 13.8 / 15.5; drawn convolutions,
// the operands from memory, 11 of 32768 and more 1.7 to 4.1 times as fast, 11 of 16384 ... 32768 0.95 to 2.1).
inline bool few_tiles_wins(long M, long N, long K, long cus, bool may_split = false) {
  return K >= 256 && few_tiles_count(M, N) <= (K < 8192 ? cus : cus / 4) &&
         !(may_split && K >= 32768);
}

// Waves that share one tile's reduction of K bytes: 2, 4, 8 or 16 for a 32 x 32 tile, -4 or -8
// for a 16 x 16 one.
int few_tiles_waves(int M, int N, int K, bool aligned);
// `aligned`: 16 | K, 16-byte aligned operands below 2 GiB.
void launch_few_tiles_fc(hipStream_t s, const FewTilesArgs& a, bool aligned, int waves);
// Extents the convolution's loader can index; the operands are 16-byte aligned and below 2 GiB.
bool few_tiles_conv_ok(int C, int K, int KH, int KW);
void launch_few_tiles_conv(hipStream_t s, FewTilesArgs a, int waves);
// Two of them of the same images in one launch.
void launch_few_tiles_pair(hipStream_t s, const FewTilesArgs& a, const FewTilesArgs& b, int waves);

// Copies of two operands with their rows of K bytes padded to Kp (a multiple of 16) with zeros:
// what brings an operand of any width to the kernels that need aligned rows.
void launch_pad_rows(hipStream_t s, const int8_t* x, long long x_rows, int8_t* x_out,
                     const int8_t* y, long long y_rows, int8_t* y_out, int K, int Kp);

}  // namespace mxq
#endif  // MXQ_FEW_TILES_H_
