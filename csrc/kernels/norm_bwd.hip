// Backward of layer norm and RMS norm (bf16, rows up to 4096 columns):
//   dx = rstd * (dy w - mean(dy w) - xhat mean(dy w xhat))
//          (RMS: rstd dy w - x rstd^3 mean(dy w x))
//   dw = sum over rows of dy xhat, db = sum of dy
//
// and, where the row went round the norm too (a residual), dx + the gradient from there,
// both rounded as apart: a pass of its own reads and writes dx once more.  In us, apart and
// here, 16384 x 768 18.2 + 13.1 and 22.9, RMS 8192 x 4096 80.9 + 31.2 and 78.7.
//
// Bound by reading x and dy and writing dx once.  A wave has a row in its
// registers between the sums and the result, and keeps its part of dw and db
// there too over all its rows, so LDS is touched once per block.

#include "../common.h"
#include "columns.h"

namespace {

struct NormBwdArgs {
  const short *dy, *x, *w;
  const short* res;              // (R, D) to be added to dx, or null
  const float *mean, *rstd;      // mean null: RMS norm
  short* dx;
  float* part;                   // [blocks][LN ? 2 : 1][D]
  long R;
  int D;
};

template <int VW> struct Vec;
template <> struct Vec<8> { using T = bf16x8; };
template <> struct Vec<4> { using T = bf16x4; };

// VW columns a load, NV loads a lane: up to 64 * VW * NV columns
template <bool LN, bool RES, int VW, int NV>
__global__ void __launch_bounds__(256)
norm_bwd_kernel(NormBwdArgs a) {
  using V = typename Vec<VW>::T;
  constexpr int SUMS = LN ? 2 : 1;
  extern __shared__ float cols[];      // [4 waves][SUMS][D]
  const int wid = threadIdx.x >> 6, l = threadIdx.x & 63;
  float dw[NV][VW] = {}, db[LN ? NV : 1][VW] = {};
  V wv[NV];
  #pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int c = (n * 64 + l) * VW;
    wv[n] = c < a.D ? *(const V*)(a.w + c) : V{};
  }
  const float inv = 1.f / (float)a.D;
  for (long row = (long)blockIdx.x * 4 + wid; row < a.R; row += (long)gridDim.x * 4) {
    V xv[NV], dv[NV], rv[RES ? NV : 1];
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = min((n * 64 + l) * VW, a.D - VW);
      xv[n] = *(const V*)(a.x + row * a.D + c);
      dv[n] = *(const V*)(a.dy + row * a.D + c);
      if constexpr (RES) rv[n] = *(const V*)(a.res + row * a.D + c);
    }
    const float mu = LN ? a.mean[row] : 0.f, rs = a.rstd[row];
    float s1 = 0.f, s2 = 0.f;
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const bool in = (n * 64 + l) * VW < a.D;
      #pragma unroll
      for (int j = 0; j < VW; ++j) {
        const float x = bf2f(xv[n][j]), d = in ? bf2f(dv[n][j]) : 0.f;
        if constexpr (LN) {
          const float xh = (x - mu) * rs, dyw = d * bf2f(wv[n][j]);
          s1 += dyw;
          s2 += dyw * xh;
          dw[n][j] += d * xh;
          db[n][j] += d;
        } else {
          s2 += d * bf2f(wv[n][j]) * x;
          dw[n][j] += d * x * rs;
        }
      }
    }
    if (LN) s1 = wave_reduce_sum(s1) * inv;
    s2 = wave_reduce_sum(s2);
    s2 = LN ? s2 * inv : rs * rs * rs * s2 / a.D;
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = (n * 64 + l) * VW;
      if (c >= a.D) continue;
      V o;
      #pragma unroll
      for (int j = 0; j < VW; ++j) {
        const float x = bf2f(xv[n][j]), d = bf2f(dv[n][j]), w = bf2f(wv[n][j]);
        if constexpr (LN) o[j] = f2bf(rs * (d * w - s1 - (x - mu) * rs * s2));
        else o[j] = f2bf(rs * d * w - x * s2);
        if constexpr (RES) o[j] = f2bf(bf2f(o[j]) + bf2f(rv[n][j]));
      }
      *(V*)(a.dx + row * a.D + c) = o;
    }
  }
  float* mine = cols + (long)wid * SUMS * a.D;
  #pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int c = (n * 64 + l) * VW;
    if (c >= a.D) continue;
    #pragma unroll
    for (int j = 0; j < VW; ++j) {
      mine[c + j] = dw[n][j];
      if (LN) mine[a.D + c + j] = db[n][j];
    }
  }
  __syncthreads();
  const int n = SUMS * a.D;
  for (int i = threadIdx.x; i < n; i += 256)
    a.part[(long)blockIdx.x * n + i] =
        cols[i] + cols[n + i] + cols[2 * n + i] + cols[3 * n + i];
}

__global__ void __launch_bounds__(1024)
norm_bwd_final_kernel(const float* __restrict__ part, short* __restrict__ dw,
                      short* __restrict__ db, int blocks, int D, int C) {
  __shared__ float acc[64][17];
  const int c = blockIdx.x * 16 + ((int)threadIdx.x & 15);
  const float s = sum_slices(part, blocks, C, c, acc);
  if (threadIdx.x >= 16 || c >= C) return;
  if (c < D) dw[c] = f2bf(s);
  else db[c - D] = f2bf(s);
}

template <bool LN, bool RES, int VW, int NV>
void launch(const NormBwdArgs& a, int blocks, hipStream_t st) {
  hipLaunchKernelGGL((norm_bwd_kernel<LN, RES, VW, NV>), dim3(blocks), dim3(256),
                     (size_t)4 * (LN ? 2 : 1) * a.D * sizeof(float), st, a);
}

template <bool LN, bool RES>
void launch(const NormBwdArgs& a, int blocks, hipStream_t st) {
  // 768 columns are 3 full loads of 4, or one and a half of 8: 16384 x 768
  // 20.7 and 25.2 us, x 520 17.5 and 22.3, 1000 x 768 7.7 and 8.2
  if (a.D <= 512) launch<LN, RES, 8, 1>(a, blocks, st);
  else if (LN && a.D <= 768) launch<LN, RES, 4, 3>(a, blocks, st);
  else if (a.D <= 1024) launch<LN, RES, 8, 2>(a, blocks, st);
  else if (a.D <= 2048) launch<LN, RES, 8, 4>(a, blocks, st);
  else launch<LN, RES, 8, 8>(a, blocks, st);
}

}  // namespace

bool norm_bwd_takes(const torch::Tensor& dy, const torch::Tensor& x,
                    const torch::Tensor& w, const c10::optional<torch::Tensor>& res) {
  auto ok = [](const torch::Tensor& t) {
    return t.scalar_type() == torch::kBFloat16 && t.is_contiguous() &&
           (size_t)t.data_ptr() % 16 == 0;
  };
  const long D = x.size(-1);
  return ok(dy) && ok(x) && ok(w) && (!res || (ok(*res) && res->sizes() == x.sizes())) &&
         D % 8 == 0 && D >= 8 && D <= 4096;
}

// dy, x, res (R, D); w (D); mean (undefined: RMS norm), rstd (R); dw, db (D)
void norm_bwd(const torch::Tensor& dy, const torch::Tensor& x,
              const torch::Tensor& w, const torch::Tensor& mean,
              const torch::Tensor& rstd, torch::Tensor& dx, torch::Tensor& dw,
              torch::Tensor& db, const c10::optional<torch::Tensor>& res,
              hipStream_t st) {
  NormBwdArgs a;
  a.R = x.size(0);
  a.D = (int)x.size(1);
  const bool ln = mean.defined();
  // More blocks leave more partial sums.  In us, with 512 and 1024, 16384 x 768
  // 21.8 and 20.9 (8192 rows 15.0 and 15.9), x 1024 25.0 and 28.9, x 2048 41.5
  // and 47.9, x 4096 160 and 180; RMS x 768 18.9 and 19.8, x 2048 36.6 and
  // 39.6.  2048 are slower throughout.
  const long most = a.D <= 1024 ? 1024 : 512;
  const int blocks = (int)std::max<long>(1, std::min(most, (a.R + 3) / 4));
  const int C = (ln ? 2 : 1) * a.D;
  auto part = torch::empty({blocks, (long)C}, rstd.options());
  a.dy = (const short*)dy.data_ptr();
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.mean = ln ? mean.data_ptr<float>() : nullptr;
  a.rstd = rstd.data_ptr<float>();
  a.res = res ? (const short*)res->data_ptr() : nullptr;
  a.dx = (short*)dx.data_ptr();
  a.part = part.data_ptr<float>();
  if (ln && a.res) launch<true, true>(a, blocks, st);
  else if (ln) launch<true, false>(a, blocks, st);
  else if (a.res) launch<false, true>(a, blocks, st);
  else launch<false, false>(a, blocks, st);
  hipLaunchKernelGGL(norm_bwd_final_kernel, dim3((C + 15) / 16), dim3(1024), 0,
                     st, a.part, (short*)dw.data_ptr(),
                     ln ? (short*)db.data_ptr() : nullptr, blocks, a.D, C);
}
