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
void big_gemm(const TileArgs& a, TileAct act, hipStream_t st);
