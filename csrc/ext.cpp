// pybind11 glue for the scaffold's gfx950 HIP kernels.
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <vector>

torch::Tensor adamw_build_meta(std::vector<torch::Tensor> masters,
                               std::vector<torch::Tensor> grads,
                               std::vector<torch::Tensor> exp_avgs,
                               std::vector<torch::Tensor> exp_avg_sqs,
                               std::vector<torch::Tensor> outs);
void fused_adamw_run(torch::Tensor meta_dev, long n, long total_vec4,
                     double lr, double beta1, double beta2, double eps,
                     double weight_decay, long step, double grad_scale,
                     bool grad_bf16, bool has_out,
                     c10::optional<torch::Tensor> step_dev);
void fused_adamw(std::vector<torch::Tensor> masters,
                 std::vector<torch::Tensor> grads,
                 std::vector<torch::Tensor> exp_avgs,
                 std::vector<torch::Tensor> exp_avg_sqs,
                 std::vector<torch::Tensor> outs, double lr, double beta1,
                 double beta2, double eps, double weight_decay, long step,
                 double grad_scale);
std::vector<torch::Tensor> layernorm_fwd(torch::Tensor x, torch::Tensor w,
                                         torch::Tensor b, double eps);
std::vector<torch::Tensor> layernorm_bwd(torch::Tensor dy, torch::Tensor x,
                                         torch::Tensor w, torch::Tensor mean,
                                         torch::Tensor rstd,
                                         c10::optional<torch::Tensor> res);
std::vector<torch::Tensor> softmax_xent_fwd(torch::Tensor logits,
                                            torch::Tensor targets);
torch::Tensor softmax_xent_bwd(torch::Tensor logits, torch::Tensor targets,
                               torch::Tensor lse, double dloss,
                               c10::optional<torch::Tensor> dloss_dev);
std::vector<torch::Tensor> rmsnorm_fwd(torch::Tensor x, torch::Tensor w,
                                       double eps);
std::vector<torch::Tensor> rmsnorm_bwd(torch::Tensor dy, torch::Tensor x,
                                       torch::Tensor w, torch::Tensor rstd,
                                       c10::optional<torch::Tensor> res);
torch::Tensor rope_apply(torch::Tensor x, torch::Tensor cos_t,
                         torch::Tensor sin_t, bool inverse,
                         c10::optional<torch::Tensor> out);
std::vector<torch::Tensor> attn_fwd(torch::Tensor q, torch::Tensor k,
                                    torch::Tensor v, bool causal);
std::vector<torch::Tensor> attn_bwd(torch::Tensor dout, torch::Tensor q,
                                    torch::Tensor k, torch::Tensor v,
                                    torch::Tensor o, torch::Tensor lse,
                                    bool causal,
                                    c10::optional<torch::Tensor> dlse,
                                    bool packed);
torch::Tensor probe_mfma(torch::Tensor A, torch::Tensor B, long which);
torch::Tensor probe_tr(torch::Tensor offsets);
torch::Tensor rccl_unique_id();
long rccl_init(long rank, long world, torch::Tensor id_bytes);
void rccl_all_reduce(long handle, torch::Tensor t);
void rccl_join(long handle);
double rccl_comm_time_ms(long handle);
void rccl_destroy(long handle);
torch::Tensor swiglu_fwd(torch::Tensor g, torch::Tensor u);
torch::Tensor swiglu_packed_fwd(torch::Tensor gu);
torch::Tensor swiglu_packed_bwd(torch::Tensor dh, torch::Tensor gu);
torch::Tensor colsum(torch::Tensor x);
void gather_into(std::vector<torch::Tensor> from, std::vector<torch::Tensor> to);
std::vector<torch::Tensor> gelu_bwd(torch::Tensor dy, torch::Tensor pre);
std::vector<torch::Tensor> swiglu_bwd(torch::Tensor dh, torch::Tensor g,
                                      torch::Tensor u);
void save_shard_pinned(std::string path, std::vector<std::string> names,
                       std::vector<torch::Tensor> tensors,
                       std::vector<std::string> meta_keys,
                       std::vector<std::string> meta_vals);
torch::Tensor weight_grad(torch::Tensor dy, torch::Tensor x);
c10::optional<torch::Tensor> wide_weight_grad(const torch::Tensor& dy, const torch::Tensor& x);
c10::optional<torch::Tensor> head_logits(const torch::Tensor& x, const torch::Tensor& w);
std::vector<torch::Tensor> head_grads(const torch::Tensor& d, const torch::Tensor& x,
                                      const torch::Tensor& w, bool want_x, bool want_w);
c10::optional<torch::Tensor> input_grad(const torch::Tensor& dy, const torch::Tensor& w);
c10::optional<torch::Tensor> residual_linear(const torch::Tensor& x, const torch::Tensor& w,
                                             const c10::optional<torch::Tensor>& bias,
                                             const torch::Tensor& res, bool last);
std::vector<torch::Tensor> linear_fwd(torch::Tensor x, torch::Tensor w,
                                      c10::optional<torch::Tensor> bias,
                                      long epilogue,
                                      c10::optional<torch::Tensor> residual);
std::vector<torch::Tensor> bn_fwd(torch::Tensor x,
                                  c10::optional<torch::Tensor> res,
                                  torch::Tensor weight, torch::Tensor bias,
                                  c10::optional<torch::Tensor> running_mean,
                                  c10::optional<torch::Tensor> running_var,
                                  double momentum, double eps, bool relu);
torch::Tensor batch_norm_act(torch::Tensor x, c10::optional<torch::Tensor> res,
                             torch::Tensor weight, torch::Tensor bias,
                             c10::optional<torch::Tensor> running_mean,
                             c10::optional<torch::Tensor> running_var,
                             double momentum, double eps, bool relu);
torch::Tensor decode_gemv(torch::Tensor x, torch::Tensor w,
                          c10::optional<torch::Tensor> bias);
c10::optional<torch::Tensor> serve_step(
    torch::Tensor tokens, torch::Tensor embed,
    c10::optional<torch::Tensor> wpe, std::vector<torch::Tensor> layers,
    std::vector<double> eps, std::vector<torch::Tensor> ks,
    std::vector<torch::Tensor> vs, c10::optional<torch::Tensor> pos, long pos0,
    c10::optional<torch::Tensor> active, c10::optional<torch::Tensor> cos_t,
    c10::optional<torch::Tensor> sin_t, std::vector<torch::Tensor> final_norm,
    torch::Tensor head, long heads, bool all);
torch::Tensor prompt_attention(torch::Tensor q, torch::Tensor k,
                               torch::Tensor v, long Sk);
torch::Tensor skinny_linear_parts(torch::Tensor x, torch::Tensor w,
                                  c10::optional<torch::Tensor> bias);
c10::optional<torch::Tensor> tile_linear(const torch::Tensor& x, const torch::Tensor& w,
                                         const c10::optional<torch::Tensor>& bias, long act,
                                         bool grad);
bool residual_takes(const torch::Tensor& x, const torch::Tensor& w, const torch::Tensor& res);
torch::Tensor skinny_linear(torch::Tensor x, torch::Tensor w,
                            c10::optional<torch::Tensor> bias,
                            c10::optional<torch::Tensor> res, long act,
                            c10::optional<torch::Tensor> norm_w,
                            c10::optional<torch::Tensor> norm_b, double eps);
torch::Tensor decode_attention(torch::Tensor qkv, torch::Tensor k,
                               torch::Tensor v, torch::Tensor pos,
                               c10::optional<torch::Tensor> active,
                               c10::optional<torch::Tensor> cos_t,
                               c10::optional<torch::Tensor> sin_t, long heads);
std::vector<torch::Tensor> bn_bwd(torch::Tensor dy, torch::Tensor x,
                                  bool has_res,
                                  c10::optional<torch::Tensor> mask,
                                  torch::Tensor weight, torch::Tensor bias,
                                  torch::Tensor mean, torch::Tensor rstd,
                                  bool relu);

// f of two tensors, or None: classes and modes that override functions see torch's product
template <typename F>
c10::optional<torch::Tensor> exact(F f, const py::object& a, const py::object& b) {
  if (at::impl::torch_function_mode_enabled() || !THPVariable_CheckExact(a.ptr()) ||
      !THPVariable_CheckExact(b.ptr()))
    return c10::nullopt;
  return f(a.cast<torch::Tensor>(), b.cast<torch::Tensor>());
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("fused_adamw", &fused_adamw, "fused multi-tensor AdamW (K1)");
  m.def("adamw_build_meta", &adamw_build_meta,
        "one-time device meta table for the cached AdamW path");
  m.def("fused_adamw_run", &fused_adamw_run,
        "AdamW step on a prebuilt meta (graph-capturable; optional device step)");
  m.def("layernorm_fwd", &layernorm_fwd, "LayerNorm forward (K2)");
  m.def("layernorm_bwd", &layernorm_bwd, "LayerNorm backward (K2)", py::arg("dy"),
        py::arg("x"), py::arg("w"), py::arg("mean"), py::arg("rstd"),
        py::arg("res") = py::none());
  m.def("softmax_xent_fwd", &softmax_xent_fwd, "softmax cross-entropy fwd (K3)");
  m.def("softmax_xent_bwd", &softmax_xent_bwd, "softmax cross-entropy bwd (K3)",
        py::arg("logits"), py::arg("targets"), py::arg("lse"),
        py::arg("dloss") = 1.0, py::arg("dloss_dev") = py::none());
  m.def("rmsnorm_fwd", &rmsnorm_fwd, "RMSNorm forward (K7)");
  m.def("rmsnorm_bwd", &rmsnorm_bwd, "RMSNorm backward (K7)", py::arg("dy"),
        py::arg("x"), py::arg("w"), py::arg("rstd"), py::arg("res") = py::none());
  m.def("rope_apply", &rope_apply, "RoPE apply/inverse (K7)", py::arg("x"),
        py::arg("cos"), py::arg("sin"), py::arg("inverse"),
        py::arg("out") = py::none());
  m.def("attn_fwd", &attn_fwd, "flash attention forward (K4)");
  m.def("attn_bwd", &attn_bwd, "flash attention backward (K4)",
        py::arg("dout"), py::arg("q"), py::arg("k"), py::arg("v"),
        py::arg("o"), py::arg("lse"), py::arg("causal"),
        py::arg("dlse") = py::none(), py::arg("packed") = false);
  m.def("probe_mfma", &probe_mfma, "MFMA fragment-layout probe (tests)");
  m.def("probe_tr", &probe_tr, "ds_read_b64_tr_b16 semantics probe (tests)");
  m.def("rccl_unique_id", &rccl_unique_id, "RCCL bootstrap id (rank 0)");
  m.def("rccl_init", &rccl_init, "init direct-RCCL bucket communicator");
  m.def("rccl_all_reduce", &rccl_all_reduce,
        "bucket SUM all-reduce on the comm stream (async)");
  m.def("rccl_join", &rccl_join, "compute stream waits comm stream");
  m.def("rccl_comm_time_ms", &rccl_comm_time_ms,
        "drain measured collective time (ms)");
  m.def("rccl_destroy", &rccl_destroy, "destroy communicator");
  m.def("swiglu_fwd", &swiglu_fwd, "fused silu(g)*u forward");
  m.def("swiglu_packed_fwd", &swiglu_packed_fwd,
        "fused SwiGLU on a packed gate|up buffer");
  m.def("swiglu_packed_bwd", &swiglu_packed_bwd,
        "packed SwiGLU backward (dgu)");
  m.def("colsum", &colsum, "bf16 column sum (bias gradients)");
  m.def("gather_into", &gather_into, "many tensors into their places");
  m.def("gelu_bwd", &gelu_bwd, "tanh-GELU backward and its column sums");
  m.def("swiglu_bwd", &swiglu_bwd, "fused SwiGLU backward (dg, du)");
  m.def("save_shard_pinned", &save_shard_pinned,
        "stream tensors to a safetensors shard via pinned D2H (C6)");
  m.def("weight_grad",
        [](py::object dy, py::object x) {
          // modes that count or replace products see torch's
          return exact([](const torch::Tensor& dy, const torch::Tensor& x) {
            return c10::impl::dispatch_mode_enabled() ? c10::nullopt
                                                      : c10::make_optional(weight_grad(dy, x));
          }, dy, x);
        },
        "dY^T X of few tiles, split over rows, or None", py::arg("dy"), py::arg("x"));
  m.def("wide_weight_grad", [](py::object dy, py::object x) { return exact(wide_weight_grad, dy, x); },
        "weight_grad where that is faster than a library, or None", py::arg("dy"),
        py::arg("x"));
  m.def("input_grad", [](py::object dy, py::object w) { return exact(input_grad, dy, w); },
        "dY W where that is faster than a library, or None", py::arg("dy"), py::arg("w"));
  m.def("residual_linear",
        [](py::object x, py::object w, py::object bias, py::object res, bool last) {
          return exact([&](const torch::Tensor& x, const torch::Tensor& w) -> c10::optional<torch::Tensor> {
            if (!THPVariable_CheckExact(res.ptr()) ||
                (!bias.is_none() && !THPVariable_CheckExact(bias.ptr())))
              return c10::nullopt;
            return residual_linear(x, w, bias.cast<c10::optional<torch::Tensor>>(),
                                   res.cast<torch::Tensor>(), last);
          }, x, w);
        },
        "x W^T + bias + res in one pass where that is faster, or None", py::arg("x"),
        py::arg("w"), py::arg("bias"), py::arg("res"), py::arg("last"));
  m.def("head_logits", [](py::object x, py::object w) { return exact(head_logits, x, w); },
        "x W^T in rows of whole lines, or None", py::arg("x"), py::arg("w"));
  m.def("head_grads", &head_grads, "dL W and dL^T x of such logits", py::arg("d"),
        py::arg("x"), py::arg("w"), py::arg("want_x"), py::arg("want_w"));
  m.def("linear_fwd", &linear_fwd,
        "MFMA linear fwd, fused bias+GELU/residual epilogue (K5)");
  m.def("bn_fwd", &bn_fwd,
        "fused bf16 NHWC BatchNorm fwd (+ReLU, +residual)",
        py::arg("x"), py::arg("res"), py::arg("weight"), py::arg("bias"),
        py::arg("running_mean"), py::arg("running_var"), py::arg("momentum"),
        py::arg("eps"), py::arg("relu"));
  m.def("batch_norm_act", &batch_norm_act,
        "bn_fwd with its gradient");
  m.def("decode_gemv", &decode_gemv,
        "decode-regime GEMV y = x W^T (+bias), B<=8",
        py::arg("x"), py::arg("w"), py::arg("bias") = py::none());
  m.def("serve_step", &serve_step,
        "a whole serving step of GPT-2 or Llama; None if not served");
  m.def("prompt_attention", &prompt_attention,
        "causal attention of S rows that end at key Sk, weights kept to 16 bits");
  m.def("skinny_linear_parts", &skinny_linear_parts,
        "sums over parts of the depth of a product of few rows", py::arg("x"),
        py::arg("w"), py::arg("bias") = py::none());
  m.def("tile_linear",
        [](py::object x, py::object w, py::object bias, long act, bool grad) {
          c10::optional<torch::Tensor> y;
          // classes and modes that override functions see torch's product
          if (at::impl::torch_function_mode_enabled()) return y;
          for (const auto* t : {&x, &w, &bias})
            if (!t->is_none() && !THPVariable_CheckExact(t->ptr())) return y;
          y = tile_linear(x.cast<torch::Tensor>(), w.cast<torch::Tensor>(),
                          bias.cast<c10::optional<torch::Tensor>>(), act, grad);
          return y;
        },
        "act(x w^T + b) of some hundred rows, or None; act: 0 none, 1 tanh-GELU, 2 erf-GELU",
        py::arg("x"), py::arg("w"), py::arg("bias") = py::none(), py::arg("act") = 0,
        py::arg("grad") = false);
  m.def("residual_takes",
        [](py::object x, py::object w, py::object res) {
          // classes and modes that override functions see torch's product
          for (const auto* t : {&x, &w, &res})
            if (!THPVariable_CheckExact(t->ptr())) return false;
          return !at::impl::torch_function_mode_enabled() &&
                 residual_takes(x.cast<torch::Tensor>(), w.cast<torch::Tensor>(),
                                res.cast<torch::Tensor>());
        },
        "whether x w^T + res or a gradient of it may be a kernel's of ours", py::arg("x"),
        py::arg("w"), py::arg("res"));
  m.def("skinny_linear", &skinny_linear,
        "product of up to 64 rows with bias, residual, GELU or SwiGLU",
        py::arg("x"), py::arg("w"), py::arg("bias") = py::none(),
        py::arg("res") = py::none(), py::arg("act") = 0,
        py::arg("norm_w") = py::none(), py::arg("norm_b") = py::none(),
        py::arg("eps") = 1e-5);
  m.def("decode_attention", &decode_attention,
        "one new token per row: rotation, cache append, attention",
        py::arg("qkv"), py::arg("k"), py::arg("v"), py::arg("pos"),
        py::arg("active"), py::arg("cos"), py::arg("sin"), py::arg("heads"));
  m.def("bn_bwd", &bn_bwd, "fused bf16 NHWC BatchNorm bwd",
        py::arg("dy"), py::arg("x"), py::arg("has_res"), py::arg("mask"),
        py::arg("weight"),
        py::arg("bias"), py::arg("mean"), py::arg("rstd"), py::arg("relu"));
}
