// Products of a few tokens with a whole weight (skinny_kernels.hip): what the dispatch in the other files needs of them.
#pragma once
#include "l8_common.h"

namespace l8 {

struct SkinnyArgs {
  const void *x, *w;    // fp8, or bf16 where the kernel quantises them
  int M, N, K;
  int64_t ldx, ldw;     // in elements
  const float *sx, *sw; // unused where the kernel quantises the operand
  int sx_row, sw_row;
  const uint16_t *bias;
  uint16_t *y;
  int64_t ldy;
  int scale_rule;
  int add;              // y = bf16(bf16(product) + y)
};

constexpr int kSkinnyMaxM = 64;
constexpr int kSkinnyAlgo = 17;  // number of these kernels among the tile configurations of l8_gemm_nt
// longest row that is quantised in registers: 12 steps of 128 elements for each of eight waves (192 registers)
constexpr int kSkinnyMaxQuantSteps = 12, kSkinnyMaxQuantK = kSkinnyMaxQuantSteps * 128 * 8;

// can the kernels serve the problem (w_bytes: 1 = fp8 weight, 2 = bf16 weight that is quantised on the way)
bool skinny_serves(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int w_bytes);
// does it pay to quantise x in the same kernel (rows of at most 4096 columns, a handful of tokens)
bool skinny_quantises_x(int64_t M, int64_t N, int64_t K, int64_t ldx, int w_bytes);
int skinny_linear(const SkinnyArgs &p, bool w_is_bf16, bool x_is_bf16, hipStream_t st);

}  // namespace l8
