// Many tensors into their places, in one launch: gradients into the flat
// buffer of a bucket.  Bound by memory; a block copies up to 32 KB of one
// tensor, 16 bytes a lane where both sides are aligned.

#include "../common.h"

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>

namespace {

constexpr int MOST = 64;               // tensors of a launch
constexpr long CHUNK = 32 * 1024;      // bytes of a block

struct GatherArgs {
  const char* from[MOST];
  char* to[MOST];
  long bytes[MOST];
  int first[MOST + 1];                 // first block of each
  int n;
};

__global__ void __launch_bounds__(256)
gather_kernel(GatherArgs a) {
  int t = 0;
  while (t + 1 < a.n && (int)blockIdx.x >= a.first[t + 1]) ++t;
  const long lo = (long)(blockIdx.x - a.first[t]) * CHUNK;
  const long n = min(CHUNK, a.bytes[t] - lo);
  const char* from = a.from[t] + lo;
  char* to = a.to[t] + lo;
  long done = 0;
  if (((size_t)from | (size_t)to) % 16 == 0) {
    done = n / 16 * 16;
    #pragma unroll 4
    for (long i = threadIdx.x * 16; i < done; i += 256 * 16)
      *(f32x4*)(to + i) = *(const f32x4*)(from + i);
  }
  // elements are of 2 bytes or more
  for (long i = done + threadIdx.x * 2; i < n; i += 256 * 2)
    *(short*)(to + i) = *(const short*)(from + i);
}

}  // namespace

// to[i] <- from[i], places in one buffer; same shape each.  One launch for all
// that are laid out alike, torch's copy for the others.
void gather_into(std::vector<torch::Tensor> from, std::vector<torch::Tensor> to) {
  TORCH_CHECK(from.size() == to.size(), "gather_into: lists differ");
  if (to.empty()) return;
  // torch's copies go by their tensors' device, whichever is current
  const auto dev = to[0].device();
  const c10::DeviceGuard guard(dev);
  const auto stream = c10::hip::getCurrentHIPStream();
  auto st = stream.stream();
  GatherArgs a;
  a.n = a.first[0] = 0;
  auto flush = [&] {
    if (a.n)
      hipLaunchKernelGGL(gather_kernel, dim3(a.first[a.n]), dim3(256), 0, st, a);
    a.n = 0;
  };
  // what lies in the buffer but not at its place is copied out before others
  // are copied in
  auto placed = [](const torch::Tensor& f, const torch::Tensor& t) {
    return f.data_ptr() == t.data_ptr() && f.strides() == t.strides() &&
           f.scalar_type() == t.scalar_type();
  };
  for (size_t i = 0; i < from.size(); ++i) {
    TORCH_CHECK(from[i].sizes() == to[i].sizes(), "gather_into: shapes differ");
    if (from[i].layout() == torch::kStrided && from[i].is_alias_of(to[i]) &&
        !placed(from[i], to[i]))
      from[i] = from[i].clone();
  }
  for (size_t i = 0; i < from.size(); ++i) {
    const auto &f = from[i], &t = to[i];
    if (!t.numel()) continue;
    if (f.layout() != torch::kStrided) {
      t.copy_(f.to_dense());
      continue;
    }
    if (placed(f, t)) continue;
    // made on another stream, it must not go back to that one's pool before it
    // has been read here (nothing to do if it is this one)
    if (f.is_cuda())
      c10::hip::HIPCachingAllocator::recordStream(f.storage().data_ptr(), stream);
    const bool alike = dev.is_cuda() && f.device() == dev && t.device() == dev &&
        f.scalar_type() == t.scalar_type() &&
        f.element_size() % 2 == 0 && f.strides() == t.strides() &&
        f.is_non_overlapping_and_dense();
    if (!alike) {
      t.copy_(f);
      continue;
    }
    if (a.n == MOST) flush();
    a.from[a.n] = (const char*)f.data_ptr();
    a.to[a.n] = (char*)t.data_ptr();
    a.bytes[a.n] = (long)f.nbytes();
    a.first[a.n + 1] = a.first[a.n] + (int)((a.bytes[a.n] + CHUNK - 1) / CHUNK);
    ++a.n;
  }
  flush();
  HIP_CHECK(hipGetLastError());
}
