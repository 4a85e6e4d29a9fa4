// One serving step of GPT-2 or Llama as a chain of launches from C++: embed,
// then per layer norm, projections, attention, feed-forward, then logits; of
// one new token per row (decoding) or of a prompt.
//
// A step of few rows is bound by its launches, not by its arithmetic: what
// can share a launch does (embedding and the first norm; residual and norm;
// bias, GELU, gate product and residual with the product before them, where
// skinny_gemm makes it), and one call from Python issues all of them.

#include "../common.h"
#include "skinny.h"
#include "tile_gemm.h"

bool decode_attention_takes(const torch::Tensor& qkv, const torch::Tensor& k,
                            const torch::Tensor& v);
torch::Tensor decode_attention(torch::Tensor qkv, torch::Tensor k,
                               torch::Tensor v, torch::Tensor pos,
                               c10::optional<torch::Tensor> active,
                               c10::optional<torch::Tensor> cos_t,
                               c10::optional<torch::Tensor> sin_t, long heads);
torch::Tensor swiglu_packed_fwd(torch::Tensor gu);
void attn_prompt(const torch::Tensor& q, const torch::Tensor& k,
                 const torch::Tensor& v, const torch::Tensor& o, int Sk,
                 hipStream_t st);

namespace {

constexpr int CHUNKS = 8;        // of 8 columns a thread: widths to 16384
constexpr long WIDEST = 256L * 8 * CHUNKS;

struct RowNormArgs {
  short* x;                      // (rows, W), read (or made) and updated
  const short* y;                // added to x first, or null
  const float* sums;             // or these, [parts][rows][W], or null
  long part;                     // elements of one of them
  int parts;
  const short *wte, *wpe;        // tok given: x = wte[tok] (+ wpe[pos])
  const long *tok, *pos;         // pos null: row r is at pos0 + r % S
  long pos0, S;
  int pos_step;
  long vocab, places;
  const short *w, *b;            // b null: RMS norm, else layer norm
  short* h;                      // null: x alone is wanted
  int W;
  float eps;
};

// A block per row, the row in registers between the sum and the result.  Of few
// rows it is the chain of waits that counts: all loads are asked for at once, those
// of the norm's weights before its sums, and none stands in a branch, behind which
// the compiler would wait for it.  2536 rows of 768 and a residual 7.0 us with the
// weights behind the sums, 5.9 so.
template <int C>
__global__ void __launch_bounds__(256)
row_norm_kernel(RowNormArgs a) {
  __shared__ float red[2][4];
  const long row = blockIdx.x;
  const int wid = threadIdx.x >> 6;
  short* x = a.x + row * a.W;
  float v[C][8];
  const short *t = nullptr, *p = nullptr;
  bool bad = false;
  if (a.tok) {
    const long id = a.tok[row], at = !a.wpe ? 0
        : a.pos ? a.pos[row * a.pos_step] : a.pos0 + row % a.S;
    bad = id < 0 || id >= a.vocab || at < 0 || (a.wpe && at >= a.places);
    t = a.wte + (bad ? 0 : id * a.W);
    p = a.wpe ? a.wpe + (bad ? 0 : at * a.W) : nullptr;
  }
  const short* from = t ? t : x;
  const short* y = a.y ? a.y + row * a.W : p;
  const short* also = y ? y : from;
  const short* bias = a.b ? a.b : a.w;
  bf16x8 e[C], f[C], w[C], b[C];
  #pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = min((c * 256 + (int)threadIdx.x) * 8, a.W - 8);
    e[c] = *(const bf16x8*)(from + i);
    f[c] = *(const bf16x8*)(also + i);
  }
  #pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = min((c * 256 + (int)threadIdx.x) * 8, a.W - 8);
    w[c] = *(const bf16x8*)(a.w + i);
    b[c] = *(const bf16x8*)(bias + i);
  }
  float s = 0.f;
  #pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = (c * 256 + threadIdx.x) * 8;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
    if (i >= a.W) continue;
    if (y)
      #pragma unroll
      for (int j = 0; j < 8; ++j) e[c][j] = f2bf(bf2f(e[c][j]) + bf2f(f[c][j]));
    if (a.sums) {
      const float* p = a.sums + row * a.W + i;
      f32x4 lo = {}, hi = {};
      #pragma unroll 4
      for (int n = 0; n < a.parts; ++n, p += a.part) {
        lo += *(const f32x4*)p;
        hi += *(const f32x4*)(p + 4);
      }
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        e[c][j] = f2bf(bf2f(e[c][j]) + lo[j]);
        e[c][4 + j] = f2bf(bf2f(e[c][4 + j]) + hi[j]);
      }
    }
    if (bad) {                           // no such row: let it show
      #pragma unroll
      for (int j = 0; j < 8; ++j) e[c][j] = 0x7fc0;
    }
    if (t || y || a.sums) *(bf16x8*)(x + i) = e[c];
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[c][j] = bf2f(e[c][j]);
      s += a.b ? v[c][j] : v[c][j] * v[c][j];
    }
  }
  if (!a.h) return;
  // over the block's four waves; waits for LDS alone
  auto total = [&](float s, int n) {
    s = wave_reduce_sum(s);
    if ((threadIdx.x & 63) == 0) red[n][wid] = s;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const f32x4 r = *(const f32x4*)red[n];
    return (r[0] + r[1]) + (r[2] + r[3]);
  };
  s = total(s, 0);
  float mean = 0.f;
  if (a.b) {
    mean = s / a.W;
    s = 0.f;
    #pragma unroll
    for (int c = 0; c < C; ++c)
      if ((c * 256 + (int)threadIdx.x) * 8 < a.W) {
        #pragma unroll
        for (int j = 0; j < 8; ++j) s += (v[c][j] - mean) * (v[c][j] - mean);
      }
    s = total(s, 1);
  }
  const float rstd = rsqrtf(s / a.W + a.eps);
  #pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = (c * 256 + threadIdx.x) * 8;
    if (i >= a.W) continue;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    u32x4 o;
    #pragma unroll
    for (int j = 0; j < 8; j += 2) {
      float h[2];
      #pragma unroll
      for (int k = 0; k < 2; ++k)
        h[k] = (v[c][j + k] - mean) * rstd * bf2f(w[c][j + k]) +
               (a.b ? bf2f(b[c][j + k]) : 0.f);
      o[j / 2] = cvt_pk_bf16(h[0], h[1]);
    }
    *(u32x4*)(a.h + row * a.W + i) = o;
  }
}

void row_norm(const RowNormArgs& a, long rows, hipStream_t st) {
  const dim3 grid((unsigned)rows), block(256);
  if (a.W <= 2048) hipLaunchKernelGGL((row_norm_kernel<1>), grid, block, 0, st, a);
  else if (a.W <= 4096) hipLaunchKernelGGL((row_norm_kernel<2>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((row_norm_kernel<CHUNKS>), grid, block, 0, st, a);
}

struct AppendArgs {
  short *qkv, *k, *v;
  long ldq, sb, sh, ss, pos0;
  int S, rows, H, G, D;          // rows of S that are appended
  const void *cos, *sin;
  int tables_bf16, turn_q;
};

// Keys (turned) and values of a prompt go to the cache, queries are turned
// where they are.  A block per token, 8 columns a thread; bound by memory.
__global__ void __launch_bounds__(256)
append_kernel(AppendArgs a) {
  const int b = blockIdx.x / a.rows, s = blockIdx.x % a.rows;
  short* row = a.qkv + ((long)b * a.S + s) * a.ldq;
  const long at = a.pos0 + s;
  const int per = a.D / 8;
  const int first = a.turn_q ? 0 : a.H * per;
  for (int c = first + threadIdx.x; c < (a.H + 2 * a.G) * per; c += 256) {
    const int head = c / per, d = c % per * 8;
    bf16x8 x = *(const bf16x8*)(row + head * a.D + d);
    if (a.cos && head < a.H + a.G) {
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long t = at * (a.D / 2) + d / 2 + i;
        const float co = a.tables_bf16 ? bf2f(((const short*)a.cos)[t])
                                       : ((const float*)a.cos)[t];
        const float si = a.tables_bf16 ? bf2f(((const short*)a.sin)[t])
                                       : ((const float*)a.sin)[t];
        const float u = bf2f(x[2 * i]), w = bf2f(x[2 * i + 1]);
        x[2 * i] = f2bf(u * co - w * si);
        x[2 * i + 1] = f2bf(u * si + w * co);
      }
    }
    short* to = row + head * a.D;
    if (head >= a.H + a.G) to = a.v + b * a.sb + (head - a.H - a.G) * a.sh + at * a.ss;
    else if (head >= a.H) to = a.k + b * a.sb + (head - a.H) * a.sh + at * a.ss;
    *(bf16x8*)(to + d) = x;
  }
}

// skinny_gemm reads x once per 16 to 64 weight rows, the library once per
// 256: with deep rows and many of them that is what counts (64 rows of
// 14336: 65 against 39 us, of 768: 6 and 7 us, 8 rows of 4096 by 28672: 47
// and 58 us)
bool few(long rows, long depth) {
  return rows <= 16 || (rows <= 64 && rows * depth <= 96 * 1024);
}

// Few rows of few heads before many keys: products of a library, in float32 over
// keys and values spread to all heads.  The line is where the flash kernel, while
// it had blocks of 256 rows, took as long; behind it weights are held in float32,
// of which the flash kernel's two parts keep 16 bits, and that stays so, although
// its blocks of 128 rows walk 1024 keys in 23 us with heads of 128 and 17 with 64
// and are ahead again for some.  In us, flash and library: 32 heads of 128, 2 rows,
// 8192 keys 188 and 232, 33 rows 193 and 330, 64 heads 187 and 452; 12 heads of 64,
// 2 rows, 8192 keys 136 and 112, 16384 267 and 126, 64 rows 279 and 214, 96 heads
// 273 and 467.  Below 5000 keys what the step's one call saves is more than the
// difference.
bool few_before_many(long heads, long S, long Sk, long D) {
  return Sk >= 5000 && (D == 64 ? heads * (S + 20) < 2750
                                : heads * (S + 45) < 3000);
}

// q (B, H, S, D), k, v (B, G, Sk, D) -> (B, S, H, D): causal, all in float32
torch::Tensor float32_attention(const torch::Tensor& q, torch::Tensor k,
                                torch::Tensor v) {
  const long rep = q.size(1) / k.size(1), S = q.size(2), Sk = k.size(2);
  if (rep > 1) {
    k = k.repeat_interleave(rep, 1);
    v = v.repeat_interleave(rep, 1);
  }
  auto s = at::matmul(q.to(at::kFloat), k.to(at::kFloat).transpose(2, 3)) *
           (1.0 / std::sqrt((double)q.size(3)));
  const auto unseen = at::ones({S, Sk}, q.options().dtype(at::kBool)).triu(Sk - S + 1);
  s.masked_fill_(unseen, -std::numeric_limits<double>::infinity());
  return at::matmul(at::softmax(s, -1), v.to(at::kFloat)).to(q.scalar_type()).transpose(1, 2);
}

}  // namespace

// tokens (B, S) -> logits (B, V) of the last token of each row, or of all,
// (B, S, V); None if this is not what the kernels are for (the caller then
// takes the step layer by layer).  layers: per layer
//   GPT-2: ln1 w, b; qkv w, b; proj w, b; ln2 w, b; fc w, b; proj w, b
//   Llama: norm w; wqkv; wo; norm w; [gate; up]; down
// wpe: GPT-2's positions (None: Llama).  pos, active (S = 1): see
// decode_attention; without pos the tokens are at pos0, pos0 + 1, ...
c10::optional<torch::Tensor> serve_step(
    torch::Tensor tokens, torch::Tensor embed,
    c10::optional<torch::Tensor> wpe, std::vector<torch::Tensor> layers,
    std::vector<double> eps, std::vector<torch::Tensor> ks,
    std::vector<torch::Tensor> vs, c10::optional<torch::Tensor> pos, long pos0,
    c10::optional<torch::Tensor> active, c10::optional<torch::Tensor> cos_t,
    c10::optional<torch::Tensor> sin_t, std::vector<torch::Tensor> final_norm,
    torch::Tensor head, long heads, bool all) {
  const bool gpt2 = wpe.has_value();
  const size_t per = gpt2 ? 12 : 6, n = ks.size();
  if (tokens.dim() != 2) return c10::nullopt;
  const long B = tokens.size(0), S = tokens.size(1), W = embed.size(-1);
  auto plain = [&](const torch::Tensor& t) {
    return t.is_cuda() && t.device() == embed.device() && t.is_contiguous() &&
           t.scalar_type() == torch::kBFloat16 &&
           (size_t)t.data_ptr() % 16 == 0;
  };
  auto is = [&](const torch::Tensor& t, long rows, long cols) {
    return plain(t) && t.dim() == (cols ? 2 : 1) && t.size(0) == rows &&
           (!cols || t.size(1) == cols);
  };
  if (!tokens.is_cuda() || tokens.scalar_type() != torch::kInt64 ||
      !tokens.is_contiguous() || B < 1 || S < 1 || n < 1 ||
      layers.size() != per * n || vs.size() != n || eps.size() != 2 * n + 1 ||
      embed.dim() != 2 || !plain(embed) || W % 8 || W > WIDEST ||
      final_norm.size() != (gpt2 ? 2u : 1u) ||
      !is(final_norm[0], W, 0) || (gpt2 && !is(final_norm[1], W, 0)) ||
      head.dim() != 2 || !is(head, head.size(0), W) ||
      (gpt2 && (wpe->dim() != 2 || !is(*wpe, wpe->size(0), W))) ||
      ks[0].dim() != 4)
    return c10::nullopt;
  const long D = ks[0].size(3), G = ks[0].size(1);
  const long qkv_n = (heads + 2 * G) * D, inner = heads * D;
  if (G < 1 || heads % G || inner % 8) return c10::nullopt;
  if (pos.has_value()) {
    if (S != 1 || !pos->is_cuda() || pos->scalar_type() != torch::kInt64 ||
        pos->dim() != 1 || !(pos->size(0) == 1 || pos->size(0) == B))
      return c10::nullopt;
  } else if (pos0 < 0 || pos0 + S > ks[0].size(2) || (S > 1 && D != 64 && D != 128) ||
             (gpt2 && pos0 + S > wpe->size(0)) ||
             (cos_t.has_value() && pos0 + S > cos_t->size(0))) {
    return c10::nullopt;
  }
  if (cos_t.has_value() &&
      !(sin_t.has_value() && cos_t->is_cuda() && sin_t->is_cuda() &&
        cos_t->is_contiguous() && sin_t->is_contiguous() && cos_t->dim() == 2 &&
        cos_t->sizes() == sin_t->sizes() && cos_t->size(1) == D / 2 &&
        cos_t->scalar_type() == sin_t->scalar_type() &&
        (cos_t->scalar_type() == torch::kFloat32 ||
         cos_t->scalar_type() == torch::kBFloat16)))
    return c10::nullopt;
  for (size_t i = 0; i < n; ++i) {
    const torch::Tensor* w = &layers[per * i];
    bool ok = ks[i].sizes() == ks[0].sizes() && ks[i].size(0) == B;
    if (gpt2) {
      const long ff = w[8].size(0);
      ok = ok && is(w[0], W, 0) && is(w[1], W, 0) && is(w[2], qkv_n, W) &&
           is(w[3], qkv_n, 0) && is(w[4], W, inner) && is(w[5], W, 0) &&
           is(w[6], W, 0) && is(w[7], W, 0) && is(w[8], ff, W) &&
           is(w[9], ff, 0) && is(w[10], W, ff) && is(w[11], W, 0) && ff % 8 == 0;
    } else {
      const long ff = w[4].size(0) / 2;
      ok = ok && is(w[0], W, 0) && is(w[1], qkv_n, W) && is(w[2], W, inner) &&
           is(w[3], W, 0) && is(w[4], 2 * ff, W) && is(w[5], W, ff) &&
           ff % 8 == 0;
    }
    if (!ok) return c10::nullopt;
  }
  long T = B * S;                  // rows of x
  const auto opt = embed.options();
  auto x = torch::empty({T, W}, opt);
  auto h = torch::empty({T, W}, opt);
  auto qkv = torch::empty({T, qkv_n}, opt);
  for (size_t i = 0; i < n; ++i)
    if (!decode_attention_takes(qkv, ks[i], vs[i])) return c10::nullopt;
  auto st = scaffold_stream();
  // where the one new token (or the last of a prompt) of each row is
  auto last_pos = [&] {
    return pos.has_value()
        ? *pos
        : torch::full({1}, pos0 + S - 1, tokens.options());
  };
  torch::Tensor at_pos;
  if (S == 1 || !all) at_pos = last_pos();

  torch::Tensor pending;           // still to be added to x: (T, W), or
                                   // (parts, T, W) float32
  const torch::Tensor* nw = nullptr;   // a norm that the next product takes
  double neps = 0;
  auto norm = [&](const torch::Tensor* w, double e, bool first, SkinnyAct act) {
    // few rows are normed by the product that reads them (which is one of
    // skinny_gemm's then)
    const bool later = w != final_norm.data() && skinny_norm_pays(T, W, act) &&
                       (first || !pending.defined());
    if (later) {
      nw = w;
      neps = e;
      if (!first) return;
    }
    RowNormArgs a = {};
    a.x = (short*)x.data_ptr();
    if (pending.defined() && pending.dim() == 3) {
      a.sums = pending.data_ptr<float>();
      a.parts = (int)pending.size(0);
      a.part = T * W;
    } else if (pending.defined()) {
      a.y = (const short*)pending.data_ptr();
    }
    if (first) {
      a.tok = tokens.data_ptr<long>();
      a.wte = (const short*)embed.data_ptr();
      a.vocab = embed.size(0);
      a.pos0 = pos0;
      a.S = S;
      if (gpt2) {
        a.wpe = (const short*)wpe->data_ptr();
        a.places = wpe->size(0);
        if (pos.has_value()) {
          a.pos = pos->data_ptr<long>();
          a.pos_step = pos->size(0) == 1 ? 0 : (int)pos->stride(0);
        }
      }
    }
    a.w = (const short*)w[0].data_ptr();
    a.b = gpt2 ? (const short*)w[1].data_ptr() : nullptr;
    a.h = later ? nullptr : (short*)h.data_ptr();
    a.W = (int)W;
    a.eps = (float)e;
    row_norm(a, T, st);
    pending = torch::Tensor();
  };
  // out = act(in w^T + b) (+ out); false: not made, take the library
  auto product = [&](const torch::Tensor& in, const torch::Tensor& w,
                     const torch::Tensor* b, torch::Tensor& out, bool add,
                     SkinnyAct act) {
    if (!few(T, in.size(1))) return false;
    if (!out.defined() || out.size(0) != T) out = torch::empty({T, w.size(0) / (act == SKINNY_SWIGLU ? 2 : 1)}, opt);
    SkinnyArgs a = {};
    a.M = (int)T;
    a.N = (int)out.size(1);
    a.K = (int)in.size(1);
    a.x = (const short*)in.data_ptr();
    a.w = (const short*)w.data_ptr();
    a.y = (short*)out.data_ptr();
    a.bias = b ? (const short*)b->data_ptr() : nullptr;
    a.res = add ? a.y : nullptr;   // read and written by the same lane
    a.ldx = a.K;
    a.ldy = a.ldr = a.N;
    if (nw && in.data_ptr() == h.data_ptr()) {   // h has not been made
      a.x = (const short*)x.data_ptr();
      a.nw = (const short*)nw[0].data_ptr();
      a.nb = gpt2 ? (const short*)nw[1].data_ptr() : nullptr;
      a.eps = (float)neps;
      nw = nullptr;
    }
    if (!skinny_takes(a)) {
      TORCH_CHECK(!a.nw, "serve_step: a norm without its product");
      return false;
    }
    skinny_gemm(a, act, st);
    return true;
  };
  // many rows: act(in w^T + b) by tiles, or undefined
  auto tiled = [&](const torch::Tensor& in, const torch::Tensor& w, const torch::Tensor* b,
                   TileAct act) {
    TileArgs a = {};
    a.M = (int)T;
    a.N = (int)w.size(0);
    a.K = (int)w.size(1);
    a.x = (const short*)in.data_ptr();
    a.w = (const short*)w.data_ptr();
    a.bias = b ? (const short*)b->data_ptr() : nullptr;
    a.ldx = a.K;
    a.ldy = a.N;
    if (!tile_takes(a, act)) return torch::Tensor();
    auto y = torch::empty({T, a.N}, opt);
    a.y = (short*)y.data_ptr();
    tile_gemm(a, act, st);
    return y;
  };
  auto lib = [&](const torch::Tensor& in, const torch::Tensor& w, const torch::Tensor* b) {
    auto y = tiled(in, w, b, TILE_NONE);
    return y.defined() ? y : b ? at::linear(in, w, *b) : at::linear(in, w);
  };
  // what is to be added to x before the next norm: in w^T + b
  auto residual = [&](const torch::Tensor& in, const torch::Tensor& w,
                      const torch::Tensor* b) {
    SkinnyArgs a = {};
    a.M = (int)T;
    a.N = (int)w.size(0);
    a.K = (int)w.size(1);
    a.x = (const short*)in.data_ptr();
    a.w = (const short*)w.data_ptr();
    a.bias = b ? (const short*)b->data_ptr() : nullptr;
    a.ldx = a.K;
    const long parts = T <= 64 && skinny_split_pays(a) ? skinny_parts(a) : 0;
    if (parts) {
      pending = torch::empty({parts, T, W}, opt.dtype(torch::kFloat32));
      skinny_split(a, pending.data_ptr<float>(), parts, st);
    } else if (!product(in, w, b, x, true, SKINNY_NONE)) {
      pending = lib(in, w, b);
    }
  };
  auto append = [&](size_t i, long rows, bool turn_q) {
    AppendArgs a = {};
    a.qkv = (short*)qkv.data_ptr();
    a.k = (short*)ks[i].data_ptr();
    a.v = (short*)vs[i].data_ptr();
    a.ldq = qkv_n;
    a.sb = ks[i].stride(0); a.sh = ks[i].stride(1); a.ss = ks[i].stride(2);
    a.pos0 = pos0;
    a.S = (int)S; a.rows = (int)rows;
    a.H = (int)heads; a.G = (int)G; a.D = (int)D;
    if (cos_t.has_value()) {
      a.cos = cos_t->data_ptr();
      a.sin = sin_t->data_ptr();
      a.tables_bf16 = cos_t->scalar_type() == torch::kBFloat16;
      a.turn_q = turn_q;
    }
    hipLaunchKernelGGL(append_kernel, dim3((unsigned)(B * rows)), dim3(256), 0, st, a);
  };
  const SkinnyAct up_act = gpt2 ? SKINNY_GELU : SKINNY_SWIGLU;
  torch::Tensor act;
  for (size_t i = 0; i < n; ++i) {
    const torch::Tensor* w = &layers[per * i];
    norm(w, eps[2 * i], i == 0, SKINNY_NONE);
    const torch::Tensor *wq = w + (gpt2 ? 2 : 1), *wo = w + (gpt2 ? 4 : 2);
    const torch::Tensor *w2 = w + (gpt2 ? 6 : 3), *up = w + (gpt2 ? 8 : 4);
    const torch::Tensor* down = w + (gpt2 ? 10 : 5);
    auto bias = [&](const torch::Tensor* t) { return gpt2 ? t + 1 : nullptr; };
    if (!product(h, *wq, bias(wq), qkv, false, SKINNY_NONE))
      qkv = lib(h, *wq, bias(wq));
    torch::Tensor o;
    if (S == 1) {
      o = decode_attention(qkv, ks[i], vs[i], at_pos, active, cos_t, sin_t, heads);
    } else if (i + 1 == n && !all) {
      // behind the last layer's keys and values only the last rows matter
      append(i, S - 1, false);
      o = decode_attention(qkv.view({B, S, qkv_n}).select(1, S - 1), ks[i],
                           vs[i], at_pos, c10::nullopt, cos_t, sin_t, heads);
      x = x.view({B, S, W}).select(1, S - 1).contiguous();
      T = B;
      h = torch::empty({T, W}, opt);
      act = torch::Tensor();
    } else {
      append(i, S, true);
      const auto q = qkv.view({B, S, heads + 2 * G, D}).narrow(2, 0, heads).transpose(1, 2);
      if (few_before_many(B * heads, S, pos0 + S, D)) {
        o = float32_attention(q, ks[i].narrow(2, 0, pos0 + S),
                              vs[i].narrow(2, 0, pos0 + S)).reshape({T, inner});
      } else {
        o = torch::empty({T, inner}, opt);
        attn_prompt(q, ks[i], vs[i], o.view({B, S, heads, D}).transpose(1, 2),
                    (int)(pos0 + S), st);
      }
    }
    residual(o, *wo, bias(wo));
    norm(w2, eps[2 * i + 1], false, up_act);
    if (act.defined() && act.size(1) != down->size(1)) act = torch::Tensor();
    if (!product(h, *up, bias(up), act, false, up_act)) {
      if (gpt2) act = tiled(h, *up, bias(up), TILE_GELU_TANH);
      if (!gpt2 || !act.defined()) {
        act = lib(h, *up, bias(up));
        act = gpt2 ? at::gelu(act, "tanh") : swiglu_packed_fwd(act);
      }
    }
    residual(act, *down, bias(down));
  }
  norm(final_norm.data(), eps[2 * n], false, SKINNY_NONE);
  torch::Tensor logits;
  if (!product(h, head, nullptr, logits, false, SKINNY_NONE))
    logits = lib(h, head, nullptr);
  HIP_CHECK(hipGetLastError());
  return all ? logits.view({B, S, head.size(0)}) : logits;
}
