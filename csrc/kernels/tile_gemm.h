// Product of some hundred rows with a weight matrix, and what may follow it; see
// tile_gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

struct TileArgs {
  const short *x, *w, *bias;     // (M, K) rows of ldx, (N, K), (N) or null
  short* y;                      // (M, N) rows of ldy
  long ldx, ldy;
  int M, N, K;
};

enum TileAct { TILE_NONE, TILE_GELU_TANH, TILE_GELU_ERF };

// Sizes and alignment it is for, where it is faster than a library
bool tile_takes(const TileArgs& a, TileAct act);
void tile_gemm(const TileArgs& a, TileAct act, hipStream_t st);

// The same for many tiles, no or the erf GELU: see big_gemm.hip
bool big_takes(const TileArgs& a, TileAct act);
bool big_alone(const TileArgs& a);        // and whether that pays for a product alone
void big_gemm(const TileArgs& a, TileAct act, hipStream_t st);
// and whether dY (M, N) W (N, K) and dY^T X, X (M, K), are that kernel's
bool input_grad_takes(long M, long N, long K);
bool weight_grad_takes(long M, long N, long K);

// Forward products that a gradient goes through.  The library (hipBLASLt of ROCm 7) was seen to
// split the depth of some deep ones (1000 x 28672 x 4096, 3000 x 28672 x 4096), whose sums then round
// otherwise, no nearer to 64 bits: through 4 layers of Llama-3-8B's width that is 2 % of the first
// step's gradients and 7 to 13 % of the next's, as much as bf16 lets either side be off, for 4 to
// 9 % of such a product.  GPT-2's, of 768 and 3072, end 0.8 % apart after two steps.  The bound
// keeps a training run the one it was with that library; no other width or version was looked at.
constexpr int BIG_DEPTH_OF_TRAINING = 3072;
