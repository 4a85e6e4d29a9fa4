// Column sum of a [R][C] bf16 matrix -> [C] (bias gradients in the
// linear backward).  torch's generic reduce ran these at ~1 TB/s, scalar
// 2-byte loads in 16 slices at a quarter of the copy rate.  This version
// is bf16x8-vectorized (G13), 4 rows' loads in flight, with a
// chip-filling slice count and a second stage whose loads are in flight
// together: 16384 x 768 in 7.8 us (18.5 with one load at a time), 16384 x
// 3072 in 18 (30).  GELU's backward takes its column sums along: 63 us at
// 16384 x 3072, 85 as two passes.

#include "../common.h"
#include "columns.h"

namespace {

typedef short bf16x8_t __attribute__((ext_vector_type(8)));

// A block has 32 columns of 8 (512 bytes of a row) and 8 rows at a time: at
// any width nearly all threads have a column.
constexpr int TILE = 32, G = 8;

// deterministic fold: per-group partials land in [g][column] slots and are
// summed in FIXED g order — an LDS atomicAdd fold would vary fp32 addition
// order run to run and break the bitwise-determinism race screen
DEVINL void fold(int C, const float (&s)[8], float (&acc)[G][TILE * 8], float* out) {
  const int t = threadIdx.x;
  #pragma unroll
  for (int j = 0; j < 8; ++j) acc[t / TILE][t % TILE * 8 + j] = s[j];
  __syncthreads();
  const int c = blockIdx.x * TILE * 8 + t;
  if (c >= C) return;
  float x = 0.f;
  #pragma unroll
  for (int g = 0; g < G; ++g) x += acc[g][t];
  out[c] = x;
}

constexpr int UN = 4;                  // rows' loads in flight

__global__ void __launch_bounds__(256)
colsum_slice_kernel(const short* __restrict__ x, float* __restrict__ mid,
                    long R, int C) {
  __shared__ float acc[G][TILE * 8];
  const int vc = blockIdx.x * TILE + threadIdx.x % TILE;
  float s[8] = {};
  if (vc < C / 8) {
    const long step = (long)gridDim.y * G;
    const short* p = x + vc * 8;
    auto add = [&](bf16x8_t v) {
      #pragma unroll
      for (int j = 0; j < 8; ++j) s[j] += bf2f(v[j]);
    };
    long r = (long)blockIdx.y * G + threadIdx.x / TILE;
    for (; r + (UN - 1) * step < R; r += UN * step) {
      bf16x8_t v[UN];
      #pragma unroll
      for (int u = 0; u < UN; ++u) v[u] = *(const bf16x8_t*)(p + (r + u * step) * C);
      #pragma unroll
      for (int u = 0; u < UN; ++u) add(v[u]);
    }
    for (; r < R; r += step) add(*(const bf16x8_t*)(p + r * C));
  }
  fold(C, s, acc, mid + (long)blockIdx.y * C);
}

// Backward of tanh-GELU, and what its result sums to by column (the bias
// gradient of the product before it) in the same pass over memory.
DEVINL float gelu_grad(float z) {
  constexpr float k = 0.7978845608028654f, a = 0.044715f;
  const float u = k * (z + a * z * z * z);
  const float t = 1.f - 2.f / (__expf(2.f * u) + 1.f);   // tanh, at both ends too
  return 0.5f * (1.f + t) + 0.5f * z * (1.f - t * t) * k * (1.f + 3.f * a * z * z);
}

__global__ void __launch_bounds__(256)
gelu_bwd_kernel(const short* __restrict__ dy, const short* __restrict__ pre,
                short* __restrict__ dpre, float* __restrict__ mid, long R,
                int C) {
  __shared__ float acc[G][TILE * 8];
  const int vc = blockIdx.x * TILE + threadIdx.x % TILE;
  float s[8] = {};
  if (vc < C / 8) {
    const long step = (long)gridDim.y * G;
    auto use = [&](long r, bf16x8_t d, bf16x8_t z) {
      bf16x8_t o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float g = bf2f(d[j]) * gelu_grad(bf2f(z[j]));
        s[j] += g;
        o[j] = f2bf(g);
      }
      *(bf16x8_t*)(dpre + r * C + vc * 8) = o;
    };
    long r = (long)blockIdx.y * G + threadIdx.x / TILE;
    for (; r + (UN - 1) * step < R; r += UN * step) {
      bf16x8_t d[UN], z[UN];
      #pragma unroll
      for (int u = 0; u < UN; ++u) {
        d[u] = *(const bf16x8_t*)(dy + (r + u * step) * C + vc * 8);
        z[u] = *(const bf16x8_t*)(pre + (r + u * step) * C + vc * 8);
      }
      #pragma unroll
      for (int u = 0; u < UN; ++u) use(r + u * step, d[u], z[u]);
    }
    for (; r < R; r += step)
      use(r, *(const bf16x8_t*)(dy + r * C + vc * 8),
          *(const bf16x8_t*)(pre + r * C + vc * 8));
  }
  fold(C, s, acc, mid + (long)blockIdx.y * C);
}

// scalar tail path for C % 8 != 0 (rare)
__global__ void __launch_bounds__(256)
colsum_slice_scalar_kernel(const short* __restrict__ x,
                           float* __restrict__ mid, long R, int C) {
  __shared__ float acc[4][64];
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int col = blockIdx.x * 64 + lane;
  const int ns = gridDim.y;
  float s = 0.f;
  if (col < C)
    for (long r = (long)blockIdx.y * 4 + wv; r < R; r += (long)ns * 4)
      s += bf2f(x[r * C + col]);
  acc[wv][lane] = s;
  __syncthreads();
  if (wv == 0 && col < C)
    mid[(long)blockIdx.y * C + col] =
        acc[0][lane] + acc[1][lane] + acc[2][lane] + acc[3][lane];
}

__global__ void __launch_bounds__(1024)
colsum_final_kernel(const float* __restrict__ mid, short* __restrict__ out,
                    int nrows, int C) {
  __shared__ float acc[64][17];
  const int c = blockIdx.x * 16 + ((int)threadIdx.x & 15);
  const float s = sum_slices(mid, nrows, C, c, acc);
  if (threadIdx.x < 16 && c < C) out[c] = f2bf(s);
}

// The same for at most 16 slices, of which 64 groups would mostly idle: 8 rows
// of 50264 take 5.4 us, 10.0 with those.
__global__ void __launch_bounds__(256)
colsum_final_few_kernel(const float* __restrict__ mid, short* __restrict__ out,
                        int nrows, int C) {
  __shared__ float acc[16][17];
  const int cl = (int)threadIdx.x & 15, g = (int)threadIdx.x >> 4;
  const int c = blockIdx.x * 16 + cl;
  acc[g][cl] = c < C && g < nrows ? mid[(long)g * C + c] : 0.f;
  __syncthreads();
  if (g || c >= C) return;
  float s = 0.f;
  #pragma unroll
  for (int j = 0; j < 16; ++j) s += acc[j][cl];
  out[c] = f2bf(s);
}

void launch_final(const torch::Tensor& mid, torch::Tensor& out, int rows, int C,
                  hipStream_t st) {
  if (rows <= 16) {
    hipLaunchKernelGGL(colsum_final_few_kernel, dim3((C + 15) / 16), dim3(256), 0,
                       st, mid.data_ptr<float>(), (short*)out.data_ptr(), rows, C);
    return;
  }
  hipLaunchKernelGGL(colsum_final_kernel, dim3((C + 15) / 16), dim3(1024), 0,
                     st, mid.data_ptr<float>(), (short*)out.data_ptr(), rows, C);
}

// blocks: enough to fill the chip, at most 256 slices.  16384 x 3072: sums 18
// us with 1024 blocks, 19 with 4096; GELU's backward 77, 66, 63 us with 512,
// 1024, 2048.
dim3 slice_grid(long R, int C, int blocks) {
  const int x = (C / 8 + TILE - 1) / TILE;
  const long ns = std::min<long>({256, std::max(1, blocks / x), (R + G - 1) / G});
  return dim3(x, (unsigned)std::max<long>(1, ns));
}

}  // namespace

torch::Tensor colsum(torch::Tensor x) {
  CHECK_CUDA(x); CHECK_CONTIG(x);
  TORCH_CHECK(x.dim() == 2 && x.scalar_type() == torch::kBFloat16);
  const long R = x.size(0);
  const int C = (int)x.size(1);
  auto out = torch::empty({C}, x.options());
  auto fopt = torch::TensorOptions().dtype(torch::kFloat32).device(x.device());
  auto stream = scaffold_stream();
  if (C % 8 == 0) {
    const dim3 grid = slice_grid(R, C, 1024);
    auto mid = torch::empty({(long)grid.y, (long)C}, fopt);
    hipLaunchKernelGGL(colsum_slice_kernel, grid, dim3(256), 0, stream,
                       (const short*)x.data_ptr(), mid.data_ptr<float>(), R, C);
    launch_final(mid, out, (int)grid.y, C, stream);
  } else {
    const int NS = R > 512 ? 16 : 1;
    auto mid = torch::empty({NS, (long)C}, fopt);
    hipLaunchKernelGGL(colsum_slice_scalar_kernel, dim3((C + 63) / 64, NS),
                       dim3(256), 0, stream, (const short*)x.data_ptr(),
                       mid.data_ptr<float>(), R, C);
    launch_final(mid, out, NS, C, stream);
  }
  HIP_CHECK(hipGetLastError());
  return out;
}

// {dpre, column sums of dpre} of y = gelu(pre), the tanh form; (R, C) bf16
std::vector<torch::Tensor> gelu_bwd(torch::Tensor dy, torch::Tensor pre) {
  CHECK_CUDA(dy); CHECK_CONTIG(dy); CHECK_CUDA(pre); CHECK_CONTIG(pre);
  TORCH_CHECK(dy.dim() == 2 && dy.sizes() == pre.sizes() &&
              dy.scalar_type() == torch::kBFloat16 &&
              pre.scalar_type() == torch::kBFloat16 && dy.size(1) % 8 == 0,
              "gelu_bwd: bf16 (R, C), C a multiple of 8");
  dy = rows16(dy);       // a slice of what cat had joined may start anywhere
  pre = rows16(pre);
  const long R = dy.size(0);
  const int C = (int)dy.size(1);
  auto dpre = torch::empty_like(pre);
  auto db = torch::empty({C}, pre.options());
  auto st = scaffold_stream();
  const dim3 grid = slice_grid(R, C, 2048);
  auto mid = torch::empty({(long)grid.y, (long)C},
                          pre.options().dtype(torch::kFloat32));
  hipLaunchKernelGGL(gelu_bwd_kernel, grid, dim3(256), 0, st,
                     (const short*)dy.data_ptr(), (const short*)pre.data_ptr(),
                     (short*)dpre.data_ptr(), mid.data_ptr<float>(), R, C);
  launch_final(mid, db, (int)grid.y, C, st);
  HIP_CHECK(hipGetLastError());
  return {dpre, db};
}
