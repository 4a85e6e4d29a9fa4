// Whether a product may go to a kernel that torch does not see.
#pragma once

#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <torch/extension.h>

// Modes that watch each call, autocast to another type, and a trace, which would hold the
// memory of the result without what was written to it.
inline bool watched() {
  return c10::impl::dispatch_mode_enabled() || at::tracer::impl::is_dispatch_enabled() ||
         (at::autocast::is_autocast_enabled(at::kCUDA) &&
          at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16);
}

// Nothing but memory on the device, of bf16: no wrapper, no batch, no tensor of zeros without
// any.
inline bool memory(const torch::Tensor& t, const torch::Device& device) {
  const auto keys = t.key_set() - c10::autograd_dispatch_keyset -
                    c10::autocast_dispatch_keyset -
                    c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
  return keys == c10::DispatchKeySet(c10::DispatchKey::CUDA) &&
         t.scalar_type() == torch::kBFloat16 && t.device() == device &&
         !t._fw_grad(0).defined();
}

// and no gradient asked of it
inline bool plain(const torch::Tensor& t, const torch::Device& device) {
  return memory(t, device) && !(at::GradMode::is_enabled() && t.requires_grad());
}
