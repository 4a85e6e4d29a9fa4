// K1 — fused multi-tensor AdamW: one launch updates every
// parameter tensor: m/v update + bias correction + decoupled decay +
// fp32-master update + bf16 working-copy refresh (K8 folded in).
//
// Pure bandwidth (28 B/element of bf16 models).  A block takes chunks of 1024 times 4
// elements of a virtual concatenation of all tensors; it looks its chunk up once, and
// a thread has the loads of four places on their way together.  Only chunks with
// several tensors in them, or a tensor's odd end, look up each place.  A block a chunk:
// 4096 blocks that walk them are 7 % slower.  GPT-2-small (124 M) in its step 583 us, 6.0 TB/s, 1.92 G
// elements of Llama's sizes 9.89 ms, 5.4 TB/s; a place a thread, looked up in 32 KB of LDS
// each, 2048 blocks, through the caches, 767 us and 11.45 ms.

#include "../common.h"

namespace {

struct AdamwArgs {
  float lr, beta1, beta2, eps, wd, bc1_inv, bc2_inv, grad_scale;
};

constexpr int MAX_TENSORS = 4096;

constexpr int CHUNK = 1024;              // places of 4 elements

// what one place needs of tensor t
struct Place {
  float *master, *m, *v;
  const void* grad;
  short* out;
};

struct Four {
  f32x4 p, m, v, g;
};

// PAST: see PAST_CACHES
template <bool BF16, bool PAST>
DEVINL Four fetch(const Place& t, long e0, float scale) {
  Four f;
  f.p = get_from<PAST>((const f32x4*)(t.master + e0));
  f.m = get_from<PAST>((const f32x4*)(t.m + e0));
  f.v = get_from<PAST>((const f32x4*)(t.v + e0));
  if constexpr (BF16) {
    const bf16x4 g = get_from<PAST>((const bf16x4*)((const short*)t.grad + e0));
    #pragma unroll
    for (int j = 0; j < 4; ++j) f.g[j] = bf2f(g[j]);
  } else {
    f.g = get_from<PAST>((const f32x4*)((const float*)t.grad + e0));
  }
  #pragma unroll
  for (int j = 0; j < 4; ++j) f.g[j] *= scale;
  return f;
}

DEVINL void update(const AdamwArgs& a, float& p, float& m, float& v, float g) {
  m = a.beta1 * m + (1.f - a.beta1) * g;
  v = a.beta2 * v + (1.f - a.beta2) * g * g;
  const float mhat = m * a.bc1_inv;
  const float vhat = v * a.bc2_inv;
  p = p * (1.f - a.lr * a.wd) - a.lr * mhat / (sqrtf(vhat) + a.eps);
}

template <bool PAST>
DEVINL void put(const AdamwArgs& a, const Place& t, long e0, Four& f, bool has_out) {
  bf16x4 o;
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    float p = f.p[j], m = f.m[j], v = f.v[j];
    update(a, p, m, v, f.g[j]);
    f.p[j] = p;
    f.m[j] = m;
    f.v[j] = v;
    o[j] = f2bf(p);
  }
  put_to<PAST>((f32x4*)(t.master + e0), f.p);
  put_to<PAST>((f32x4*)(t.m + e0), f.m);
  put_to<PAST>((f32x4*)(t.v + e0), f.v);
  if (has_out) *(bf16x4*)(t.out + e0) = o;
}

// meta layout (int64 words): [0..n] starts_vec4 cumsum; then per-array
// pointer blocks: master[n], grad[n], m[n], v[n], out[n], numel[n]
DEVINL Place place_of(const long* meta, int n, int t) {
  const long* list = meta + (n + 1);
  return {(float*)list[t], (float*)list[2l * n + t], (float*)list[3l * n + t],
          (const void*)list[n + t], (short*)list[4l * n + t]};
}

// place vi, of tensor t
template <bool BF16>
DEVINL void one(const AdamwArgs& a, const long* meta, int n, int t, long vi, bool has_out) {
  const Place at = place_of(meta, n, t);
  const long e0 = (vi - meta[t]) * 4, numel = meta[n + 1 + 5l * n + t];
  if (e0 + 4 <= numel) {
    Four f = fetch<BF16, false>(at, e0, a.grad_scale);
    put<false>(a, at, e0, f, has_out);
    return;
  }
  for (long e = e0; e < numel; ++e) {
    const float g = (BF16 ? bf2f(((const short*)at.grad)[e])
                          : ((const float*)at.grad)[e]) * a.grad_scale;
    update(a, at.master[e], at.m[e], at.v[e], g);
    if (has_out) at.out[e] = f2bf(at.master[e]);
  }
}

DEVINL void at_step(AdamwArgs& a, const int* step_dev) {
  if (step_dev == nullptr) return;
  // hipGraph-replay path: the step lives on DEVICE (incremented by a
  // captured op), so bias corrections stay exact under replay where
  // host-baked args would freeze at the capture step.
  const float s = (float)*step_dev;
  a.bc1_inv = 1.0f / (1.0f - __powf(a.beta1, s));
  a.bc2_inv = 1.0f / (1.0f - __powf(a.beta2, s));
}

// Few elements, or many tensors of few: a place a thread, looked up in LDS.  In us, so, in
// chunks, and (before) so with 32 KB of LDS and types looked at in each: 268 thousand elements
// in 6 tensors 4.9 and 7.8; 1.2 M in one 8.3, 10.6 and 8.9, 4 M 19.8, 18.5 and 20.3; 2.6 M in 48
// of all sizes 15.2, 17.5 and 16.6, 4.1 M in 53 20.9, 22.0 and 22.9; 4096 tensors of 7 8.6 and 20.7,
// 900 of 4097 22.3, 20.1 and 24.5.  The line is where chunks are no slower than before.
constexpr long FEW = 1 << 20;            // places

template <bool BF16>
__global__ void __launch_bounds__(256)
adamw_few_kernel(const long* __restrict__ meta, int n, long total_vec4,
                 AdamwArgs a, int has_out, const int* __restrict__ step_dev) {
  __shared__ long s_starts[MAX_TENSORS + 1];
  for (int i = threadIdx.x; i <= n; i += blockDim.x) s_starts[i] = meta[i];
  __syncthreads();
  at_step(a, step_dev);
  for (long vi = (long)blockIdx.x * blockDim.x + threadIdx.x; vi < total_vec4;
       vi += grid_stride()) {
    // largest t with s_starts[t] <= vi
    int lo = 0, hi = n - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_starts[mid] <= vi) lo = mid; else hi = mid - 1;
    }
    one<BF16>(a, meta, n, lo, vi, has_out);
  }
}

// More places than this (16.8 million elements, of which a step reads and writes 268 MB and more):
// moments and masters go past the memory-side cache, of 256 MB, both ways, so that nothing is
// written back before something is read.  The new weights go through it.  Where the line lies
// depends on what the cache holds.  Through it and past it, in us, of bf16 gradients: step upon
// step 10 million 45 and 53, 17 million 88 and 93, 22 million 117 and 115, 25 million 137 and 120,
// 60 million 320 and 265, 124 million 700 and 565 (6.2 TB/s), 400 million 2354 and 2186; but
// behind 1.2 GB that were written, as a backward leaves it, 17 million 116 and 100, 20 million 130 and
// 116.  With the stores alone past it 717 for 124 million, with the loads alone 678.
constexpr long PAST_CACHES = 4 << 20;    // places

template <bool BF16, bool PAST>
__global__ void __launch_bounds__(256)
adamw_mt_kernel(const long* __restrict__ meta, int n, long total_vec4,
                AdamwArgs a, int has_out, const int* __restrict__ step_dev) {
  at_step(a, step_dev);
  // largest t with meta[t] <= vi, for the whole wave: a lane looks at one of 64, then
  // at one behind the last of those: a step has to be one look, of 64 lanes
  static_assert(MAX_TENSORS <= 64 * 64, "a lane looks at one");
  const int l = threadIdx.x & 63, step = (n + 63) / 64;
  auto find = [&](long vi) {
    int t = (__popcll(__ballot(l * step < n && meta[min(l * step, n - 1)] <= vi)) - 1) * step;
    const int at = t + 1 + l;
    t += __popcll(__ballot(1 + l < step && at < n && meta[min(at, n - 1)] <= vi));
    return __builtin_amdgcn_readfirstlane(t);
  };
  const long chunks = (total_vec4 + CHUNK - 1) / CHUNK;
  for (long c = blockIdx.x; c < chunks; c += gridDim.x) {
    const int t = find(c * CHUNK);
    const long first = c * CHUNK - meta[t];
    if ((first + CHUNK) * 4 <= meta[n + 1 + 5l * n + t]) {
      const Place at = place_of(meta, n, t);
      const long e0 = (first + threadIdx.x) * 4;
      Four f[4];
      #pragma unroll
      for (int u = 0; u < 4; ++u) f[u] = fetch<BF16, PAST>(at, e0 + u * 1024, a.grad_scale);
      #pragma unroll
      for (int u = 0; u < 4; ++u) put<PAST>(a, at, e0 + u * 1024, f[u], has_out);
      continue;
    }
    const long end = min(total_vec4, (c + 1) * CHUNK);
    const int last = find(end - 1);
    for (long vi = c * CHUNK + threadIdx.x; vi < end; vi += 256) {
      int lo = t, hi = last;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (meta[mid] <= vi) lo = mid; else hi = mid - 1;
      }
      one<BF16>(a, meta, n, lo, vi, has_out);
    }
  }
}

}  // namespace

// Build the device meta table ONCE (pointers are stable across steps:
// grads are bucket views, masters/moments never reallocate) so the hot
// step — and a hipGraph capture of it — carries no H2D copy.
torch::Tensor adamw_build_meta(std::vector<torch::Tensor> masters,
                               std::vector<torch::Tensor> grads,
                               std::vector<torch::Tensor> exp_avgs,
                               std::vector<torch::Tensor> exp_avg_sqs,
                               std::vector<torch::Tensor> outs) {
  const int n = (int)masters.size();
  TORCH_CHECK(n > 0 && n <= MAX_TENSORS, "fused_adamw: 1..4096 tensors, got ", n);
  const bool has_out = !outs.empty();
  TORCH_CHECK(!has_out || (int)outs.size() == n);

  std::vector<long> meta;
  meta.reserve((size_t)n * 7 + 1);
  long cum = 0;
  for (int i = 0; i < n; ++i) {
    meta.push_back(cum);
    cum += (masters[i].numel() + 3) / 4;
  }
  meta.push_back(cum);
  auto push_ptrs = [&](std::vector<torch::Tensor>& ts) {
    for (int i = 0; i < n; ++i) meta.push_back((long)ts[i].data_ptr());
  };
  push_ptrs(masters);
  push_ptrs(grads);
  push_ptrs(exp_avgs);
  push_ptrs(exp_avg_sqs);
  if (has_out) push_ptrs(outs);
  else for (int i = 0; i < n; ++i) meta.push_back(0);
  for (int i = 0; i < n; ++i) meta.push_back(masters[i].numel());

  auto opts = torch::TensorOptions().dtype(torch::kInt64);
  auto meta_cpu = torch::from_blob(meta.data(), {(long)meta.size()}, opts).clone();
  return meta_cpu.to(masters[0].device());
}

void fused_adamw_run(torch::Tensor meta_dev, long n, long total_vec4,
                     double lr, double beta1, double beta2, double eps,
                     double weight_decay, long step, double grad_scale,
                     bool grad_bf16, bool has_out,
                     c10::optional<torch::Tensor> step_dev) {
  AdamwArgs a;
  a.lr = (float)lr;
  a.beta1 = (float)beta1;
  a.beta2 = (float)beta2;
  a.eps = (float)eps;
  a.wd = (float)weight_decay;
  a.bc1_inv = (float)(1.0 / (1.0 - std::pow(beta1, (double)step)));
  a.bc2_inv = (float)(1.0 / (1.0 - std::pow(beta2, (double)step)));
  a.grad_scale = (float)grad_scale;

  const int* sd = nullptr;
  if (step_dev.has_value()) {
    TORCH_CHECK(step_dev->scalar_type() == torch::kInt32 && step_dev->is_cuda());
    sd = step_dev->data_ptr<int>();
  }
  const bool few = total_vec4 < FEW;
  const dim3 grid(few ? capped_blocks(total_vec4, 256, 2048)
                      // below 2^32 threads
                      : (int)std::min<long>((total_vec4 + CHUNK - 1) / CHUNK, 1 << 23));
  auto stream = scaffold_stream();
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, meta_dev.data_ptr<long>(), (int)n,
                       total_vec4, a, has_out ? 1 : 0, sd);
  };
  if (few) grad_bf16 ? run(adamw_few_kernel<true>) : run(adamw_few_kernel<false>);
  else if (total_vec4 < PAST_CACHES)
    grad_bf16 ? run(adamw_mt_kernel<true, false>) : run(adamw_mt_kernel<false, false>);
  else grad_bf16 ? run(adamw_mt_kernel<true, true>) : run(adamw_mt_kernel<false, true>);
  HIP_CHECK(hipGetLastError());
}

void fused_adamw(std::vector<torch::Tensor> masters,
                 std::vector<torch::Tensor> grads,
                 std::vector<torch::Tensor> exp_avgs,
                 std::vector<torch::Tensor> exp_avg_sqs,
                 std::vector<torch::Tensor> outs,  // bf16 working copies or empty
                 double lr, double beta1, double beta2, double eps,
                 double weight_decay, long step, double grad_scale) {
  const int n = (int)masters.size();
  TORCH_CHECK(n > 0, "fused_adamw: empty tensor list");
  long cum = 0;
  for (int i = 0; i < n; ++i) cum += (masters[i].numel() + 3) / 4;
  auto meta_dev = adamw_build_meta(masters, grads, exp_avgs, exp_avg_sqs, outs);
  fused_adamw_run(meta_dev, n, cum, lr, beta1, beta2, eps, weight_decay, step,
                  grad_scale, grads[0].scalar_type() == torch::kBFloat16,
                  !outs.empty(), c10::nullopt);
}
