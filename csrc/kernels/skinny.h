// Product of few rows with a weight matrix, and what may follow it; see
// skinny_gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

struct SkinnyArgs {
  const short *x, *w;            // (M, K) rows of ldx, (N or 2N, K)
  long ldx;
  int M, N, K;
  int fours;                     // skinny_gemm: y, bias and res lie for 8-byte access
  const short *nw, *nb;          // x is normed first: layer norm with nb, else RMS
                                 // norm; null: as it is
  const short *bias, *res;       // (N) or null; (M, N) rows of ldr or null
  short *y;                      // (M, N) rows of ldy
  long ldr, ldy;
  float eps;                     // of the norm
};

enum SkinnyAct {
  SKINNY_NONE,                   // y = x w^T + bias + res
  SKINNY_GELU,                   // gelu(x w^T + bias), the tanh form
  SKINNY_SWIGLU,                 // silu(x g^T) * (x u^T), w = [g; u]
};

// M up to 64, K a multiple of 8, x and w rows 16-byte aligned
bool skinny_takes(const SkinnyArgs& a);
bool skinny_norms(long M, long K);     // whether it may have a norm
bool skinny_norm_pays(long M, long K, SkinnyAct act);   // against a launch of its own
void skinny_gemm(SkinnyArgs a, SkinnyAct act, hipStream_t st);

// The same without act, res or norm, the depth split over `parts` groups of
// blocks whose sums, (parts, M, N) float32 with the bias in the first, the
// reader adds.  0: not what it is for.
long skinny_parts(const SkinnyArgs& a);
bool skinny_split_pays(const SkinnyArgs& a);   // against whole depths, the library
void skinny_split(const SkinnyArgs& a, float* sums, long parts, hipStream_t st);
