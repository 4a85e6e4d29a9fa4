// Decode attention over a dense key/value cache (bf16): one new token per
// row, every row at its own depth.
//
// One launch takes the packed projections [q heads | k heads | v heads] of
// the new tokens, turns q and k, appends k and v to the cache and attends:
// the block that owns the token's place uses the new key and value from
// registers and stores them, the others read what is cached.
//
// What bounds it is reading the cache once.  A block has one kv head of one
// row, up to 4 query heads that share it, and one span of the keys; a cached
// row goes from memory to the registers that use it (a lane has 8 columns of
// a key, 16 lanes a key of 128), so there is no LDS traffic and no barrier
// in the loop, and each group of lanes keeps a running maximum of its own
// until the end.  Spans exist so that few rows fill the chip; depths are
// read on the device, and blocks behind a row's depth end at once, so the
// grid is the same at every depth and a step can be captured.  Scores,
// softmax, weights and sums are float32.

#include "../common.h"

namespace {

// "no key yet", base-2 scores.  What is not above it weighs nothing, which of
// a key's scores only -inf is: the comparisons below let NaN pass, so that it
// shows in the row.
constexpr float NONE = -3.4028234663852886e38f;

struct DecodeArgs {
  const short *qkv;
  short *k, *v;
  long ldq, sb, sh, ss;          // of qkv rows; of the cache (k and v alike)
  const long *pos;               // one per row, or one for all (pos_step 0)
  const long *active;            // 0: leave the row alone; null: all active
  int pos_step;
  const void *cos, *sin;         // (positions, D/2); null: nothing turns
  int tables_bf16;
  float *part;                   // [B*H][spans][D + 2]
  short *out;                    // [B][H*D]
  int B, H, G, spans, span, waves;
  long limit;                    // positions that exist: cache and tables
  float scale2;                  // of scores, times log2(e)
};

// sum over the lanes of a group of N (8, 16: within a row of 16 lanes)
template <int N> DEVINL float group_sum(float x) {
  auto dpp = [](float v, auto ctrl) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
        0, i, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x += dpp(x, std::integral_constant<int, 0xB1>{});    // lane ^ 1
  x += dpp(x, std::integral_constant<int, 0x4E>{});    // lane ^ 2
  if constexpr (N >= 8) x += dpp(x, std::integral_constant<int, 0x141>{});
  if constexpr (N >= 16) x += dpp(x, std::integral_constant<int, 0x140>{});
  return x;
}

DEVINL float table(const void* t, int is_bf16, long i) {
  return is_bf16 ? bf2f(((const short*)t)[i]) : ((const float*)t)[i];
}

// 8 columns of a head, from column 8*c on, pairs (2i, 2i+1) turned and
// rounded as the cache holds them
template <int D>
DEVINL bf16x8 turned(const DecodeArgs& a, const short* p, int c, long pos) {
  bf16x8 x = *(const bf16x8*)(p + 8 * c);
  if (!a.cos) return x;
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long t = pos * (D / 2) + 4 * c + i;
    const float co = table(a.cos, a.tables_bf16, t);
    const float si = table(a.sin, a.tables_bf16, t);
    const float u = bf2f(x[2 * i]), w = bf2f(x[2 * i + 1]);
    x[2 * i] = f2bf(u * co - w * si);
    x[2 * i + 1] = f2bf(u * si + w * co);
  }
  return x;
}

// D: head size; R: query heads of a block; WAVES: of a block
template <int D, int R, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
decode_attn_kernel(DecodeArgs a) {
  constexpr int LPK = D / 8;            // lanes per key
  constexpr int KPI = 64 / LPK;         // keys per load of a wave
  constexpr int U = 4;                  // loads in flight
  constexpr int TILE = KPI * U;
  __shared__ float sm[WAVES][R][2], so[WAVES][R][D];

  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int g = l / LPK, c = l % LPK;   // key within a load, column chunk
  const int rep = a.H / a.G, chunks = (rep + R - 1) / R;
  const int s = blockIdx.x;
  const int b = blockIdx.y / (a.G * chunks);
  const int kv = blockIdx.y / chunks % a.G, ch = blockIdx.y % chunks;
  const int h0 = kv * rep + ch * R, heads = min(R, rep - ch * R);

  const long pos = a.pos[(long)b * a.pos_step];
  const bool on = (!a.active || a.active[b]) && pos >= 0 && pos < a.limit;
  const int lo = s * a.span;
  if (!on) {
    // nothing is written for the row; a place outside the cache shows
    if (s == 0 && w == 0)
      for (int i = l; i < heads * D; i += 64)
        a.out[(long)b * a.H * D + (long)h0 * D + i] =
            !a.active || a.active[b] ? 0x7fc0 : 0;
    return;
  }
  const int p = (int)pos;
  if (lo > p) return;
  const int hi = min(p, lo + a.span);   // cached keys [lo, hi)
  const bool own = p < lo + a.span;     // the new key's place is here

  short* kc = a.k + b * a.sb + kv * a.sh + 8 * c;
  short* vc = a.v + b * a.sb + kv * a.sh + 8 * c;

  // the next tile's rows are on their way while one is used; places behind
  // the last key repeat it and do not count
  const int last = max(hi - 1, 0);
  auto fetch = [&](bf16x8 (&kk)[U], bf16x8 (&vv)[U], int j0) {
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      const long at = (long)min(j0 + u * KPI + g, last) * a.ss;
      kk[u] = *(const bf16x8*)(kc + at);
      vv[u] = *(const bf16x8*)(vc + at);
    }
  };
  bf16x8 k0[U], v0[U], k1[U], v1[U];
  int j = lo + w * TILE;
  if (j < hi) fetch(k0, v0, j);

  const short* row = a.qkv + (long)b * a.ldq;
  float q[R][8];
  #pragma unroll
  for (int r = 0; r < R; ++r) {
    const bf16x8 t = turned<D>(a, row + (h0 + min(r, heads - 1)) * D, c, p);
    #pragma unroll
    for (int i = 0; i < 8; ++i) q[r][i] = bf2f(t[i]) * a.scale2;
  }
  float m[R], sum[R], o[R][8];
  #pragma unroll
  for (int r = 0; r < R; ++r) {
    m[r] = NONE;
    sum[r] = 0.f;
    #pragma unroll
    for (int i = 0; i < 8; ++i) o[r][i] = 0.f;
  }
  auto take = [&](const bf16x8 (&kk)[U], bf16x8 (&vv)[U], int j0) {
    // no weight makes an infinite value nothing, so those of the repeated
    // places go; only a row's last tile has some
    if (j0 + TILE > hi) {
      #pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u * KPI + g >= hi) vv[u] = bf16x8{};
    }
    float sc[U][R];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      float kf[8];
      #pragma unroll
      for (int i = 0; i < 8; ++i) kf[i] = bf2f(kk[u][i]);
      const bool see = j0 + u * KPI + g < hi;
      #pragma unroll
      for (int r = 0; r < R; ++r) {
        float d = 0.f;
        #pragma unroll
        for (int i = 0; i < 8; ++i) d = fmaf(q[r][i], kf[i], d);
        d = group_sum<LPK>(d);
        sc[u][r] = see ? d : NONE;
      }
    }
    #pragma unroll
    for (int r = 0; r < R; ++r) {
      float t = m[r];
      #pragma unroll
      for (int u = 0; u < U; ++u) t = fmaxf(t, sc[u][r]);
      const float f = __builtin_amdgcn_exp2f(m[r] - t);
      m[r] = t;
      sum[r] *= f;
      #pragma unroll
      for (int i = 0; i < 8; ++i) o[r][i] *= f;
    }
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      float vf[8];
      #pragma unroll
      for (int i = 0; i < 8; ++i) vf[i] = bf2f(vv[u][i]);
      #pragma unroll
      for (int r = 0; r < R; ++r) {
        // a score of NONE is no key, also where the maximum is none yet
        const float e = sc[u][r] <= NONE
            ? 0.f : __builtin_amdgcn_exp2f(sc[u][r] - m[r]);
        sum[r] += e;
        #pragma unroll
        for (int i = 0; i < 8; ++i) o[r][i] = fmaf(e, vf[i], o[r][i]);
      }
    }
  };
  for (; j < hi; j += 2 * WAVES * TILE) {
    const int next = j + WAVES * TILE;
    if (next < hi) fetch(k1, v1, next);
    take(k0, v0, j);
    if (next >= hi) break;
    if (next + WAVES * TILE < hi) fetch(k0, v0, next + WAVES * TILE);
    take(k1, v1, next);
  }
  // the new token, by the last wave's first group of lanes
  if (own && w == WAVES - 1) {
    const bf16x8 nk = turned<D>(a, row + (a.H + kv) * D, c, p);
    bf16x8 nv = *(const bf16x8*)(row + (a.H + a.G + kv) * D + 8 * c);
    if (g == 0 && ch == 0) {
      *(bf16x8*)(kc + (long)p * a.ss) = nk;
      *(bf16x8*)(vc + (long)p * a.ss) = nv;
    }
    if (g != 0) nv = bf16x8{};
    #pragma unroll
    for (int r = 0; r < R; ++r) {
      float d = 0.f;
      #pragma unroll
      for (int i = 0; i < 8; ++i) d = fmaf(q[r][i], bf2f(nk[i]), d);
      d = group_sum<LPK>(d);
      if (g != 0) d = NONE;
      const float t = fmaxf(m[r], d), f = __builtin_amdgcn_exp2f(m[r] - t);
      const float e = d <= NONE ? 0.f : __builtin_amdgcn_exp2f(d - t);
      m[r] = t;
      sum[r] = sum[r] * f + e;
      #pragma unroll
      for (int i = 0; i < 8; ++i) o[r][i] = o[r][i] * f + e * bf2f(nv[i]);
    }
  }
  // groups of lanes, then waves
  #pragma unroll
  for (int r = 0; r < R; ++r) {
    #pragma unroll
    for (int x = LPK; x < 64; x *= 2) {
      const float mo = __shfl_xor(m[r], x, 64), t = fmaxf(m[r], mo);
      const float f = __builtin_amdgcn_exp2f(m[r] - t);
      const float fo = __builtin_amdgcn_exp2f(mo - t);
      sum[r] = sum[r] * f + __shfl_xor(sum[r], x, 64) * fo;
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        o[r][i] = o[r][i] * f + __shfl_xor(o[r][i], x, 64) * fo;
      m[r] = t;
    }
    if (g == 0) {
      #pragma unroll
      for (int i = 0; i < 8; ++i) so[w][r][8 * c + i] = o[r][i];
      if (c == 0) {
        sm[w][r][0] = m[r];
        sm[w][r][1] = sum[r];
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < heads * D; i += 64 * WAVES) {
    const int r = i / D, d = i % D, h = h0 + r;
    float t = NONE, den = 0.f, num = 0.f;
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) t = fmaxf(t, sm[x][r][0]);
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) {
      const float f = __builtin_amdgcn_exp2f(sm[x][r][0] - t);
      den += f * sm[x][r][1];
      num += f * so[x][r][d];
    }
    if (a.spans == 1) {
      a.out[((long)b * a.H + h) * D + d] = f2bf(num / den);
      continue;
    }
    float* part = a.part + (((long)b * a.H + h) * a.spans + s) * (D + 2);
    part[d] = num;
    if (d == 0) {
      part[D] = t;
      part[D + 1] = den;
    }
  }
}

// a block per head: its spans' sums, weighted by their maxima
template <int D>
__global__ void __launch_bounds__(D < 64 ? 64 : D)
decode_merge_kernel(DecodeArgs a) {
  const long bh = blockIdx.x;
  const int b = (int)(bh / a.H), d = threadIdx.x;
  const long pos = a.pos[(long)b * a.pos_step];
  if ((a.active && !a.active[b]) || pos < 0 || pos >= a.limit || d >= D) return;
  const int n = (int)pos / a.span + 1;
  const float* part = a.part + bh * a.spans * (D + 2);
  float t = NONE, den = 0.f, num = 0.f;
  #pragma unroll 4
  for (int s = 0; s < n; ++s) t = fmaxf(t, part[s * (D + 2) + D]);
  #pragma unroll 4
  for (int s = 0; s < n; ++s) {
    const float* p = part + s * (D + 2);
    const float f = __builtin_amdgcn_exp2f(p[D] - t);
    den += f * p[D + 1];
    num += f * p[d];
  }
  a.out[bh * D + d] = f2bf(num / den);
}

template <int D, int R>
void launch(const DecodeArgs& a, hipStream_t st) {
  const int chunks = (a.H / a.G + R - 1) / R;
  const dim3 grid(a.spans, a.B * a.G * chunks);
  if (a.waves == 8)
    hipLaunchKernelGGL((decode_attn_kernel<D, R, 8>), grid, dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((decode_attn_kernel<D, R, 4>), grid, dim3(256), 0, st, a);
  if (a.spans > 1)
    hipLaunchKernelGGL((decode_merge_kernel<D>), dim3(a.B * a.H),
                       dim3(D < 64 ? 64 : D), 0, st, a);
}

template <int D>
void launch(const DecodeArgs& a, hipStream_t st) {
  const int rep = a.H / a.G;
  if (rep == 1) launch<D, 1>(a, st);
  else if (rep == 2) launch<D, 2>(a, st);
  else launch<D, 4>(a, st);
}

}  // namespace

// What decode_attention takes: see there.
bool decode_attention_takes(const torch::Tensor& qkv, const torch::Tensor& k,
                            const torch::Tensor& v) {
  const long D = k.dim() == 4 ? k.size(3) : 0;
  return qkv.is_cuda() && k.is_cuda() && v.is_cuda() && qkv.dim() == 2 &&
         (D == 32 || D == 64 || D == 128) && v.sizes() == k.sizes() &&
         v.strides() == k.strides() &&
         qkv.scalar_type() == torch::kBFloat16 &&
         k.scalar_type() == torch::kBFloat16 &&
         v.scalar_type() == torch::kBFloat16 && qkv.stride(1) == 1 &&
         k.stride(3) == 1 && qkv.stride(0) % 8 == 0 && k.stride(0) % 8 == 0 &&
         k.stride(1) % 8 == 0 && k.stride(2) % 8 == 0 &&
         (size_t)qkv.data_ptr() % 16 == 0 && (size_t)k.data_ptr() % 16 == 0 &&
         (size_t)v.data_ptr() % 16 == 0;
}

// qkv (B, (H + 2G) * D) bf16 rows; k, v (B, G, L, D) of one layer; pos (B)
// or (1) int64.  Returns (B, H * D).
torch::Tensor decode_attention(torch::Tensor qkv, torch::Tensor k,
                               torch::Tensor v, torch::Tensor pos,
                               c10::optional<torch::Tensor> active,
                               c10::optional<torch::Tensor> cos_t,
                               c10::optional<torch::Tensor> sin_t, long heads) {
  CHECK_CUDA(pos);
  TORCH_CHECK(decode_attention_takes(qkv, k, v), "decode_attention: bf16 on "
              "the GPU, heads of 32, 64 or 128, rows 16-byte aligned");
  DecodeArgs a;
  a.B = (int)qkv.size(0);
  a.H = (int)heads;
  a.G = (int)k.size(1);
  const int L = (int)k.size(2);
  a.limit = L;
  const int D = (int)k.size(3);
  TORCH_CHECK(a.G > 0 && a.H % a.G == 0 && k.size(0) == a.B &&
              qkv.size(1) == (long)(a.H + 2 * a.G) * D,
              "decode_attention: heads");
  TORCH_CHECK(pos.scalar_type() == torch::kInt64 && pos.dim() == 1 &&
              (pos.size(0) == a.B || pos.size(0) == 1),
              "decode_attention: pos is (rows,) int64");
  a.pos_step = pos.size(0) == 1 ? 0 : (int)pos.stride(0);
  a.active = nullptr;
  if (active.has_value()) {
    TORCH_CHECK(active->is_cuda() && active->scalar_type() == torch::kInt64 &&
                active->is_contiguous() && active->numel() == a.B,
                "decode_attention: active is (rows,) int64");
    a.active = active->data_ptr<long>();
  }
  a.cos = a.sin = nullptr;
  a.tables_bf16 = 0;
  if (cos_t.has_value()) {
    TORCH_CHECK(sin_t.has_value() && cos_t->is_cuda() && sin_t->is_cuda() &&
                cos_t->is_contiguous() && sin_t->is_contiguous() &&
                cos_t->sizes() == sin_t->sizes() &&
                cos_t->scalar_type() == sin_t->scalar_type() &&
                (cos_t->scalar_type() == torch::kFloat32 ||
                 cos_t->scalar_type() == torch::kBFloat16) &&
                cos_t->dim() == 2 && cos_t->size(1) == D / 2,
                "decode_attention: rotary tables");
    a.limit = std::min<long>(L, cos_t->size(0));
    a.cos = cos_t->data_ptr();
    a.sin = sin_t->data_ptr();
    a.tables_bf16 = cos_t->scalar_type() == torch::kBFloat16;
  }
  a.qkv = (const short*)qkv.data_ptr();
  a.k = (short*)k.data_ptr();
  a.v = (short*)v.data_ptr();
  a.pos = pos.data_ptr<long>();
  a.ldq = qkv.stride(0);
  a.sb = k.stride(0); a.sh = k.stride(1); a.ss = k.stride(2);
  a.scale2 = 1.4426950408889634f / std::sqrt((float)D);
  auto out = torch::empty({a.B, (long)a.H * D}, qkv.options());
  a.out = (short*)out.data_ptr();
  if (a.B == 0) return out;
  // Spans of whole 64s.  With 256 pairs of a row and a kv head or more, 512
  // blocks of 4 waves fill the chip (64 rows of 8 kv heads to 4096 deep: 155
  // us in one span each, 162 us with 8 waves); with fewer, 256 blocks of 8
  // waves (8 rows to 2048: 26 us, 35 us as 1024 blocks of 4).  A cache that
  // 8 waves walk in 4 steps is one span, which saves the merge (8 rows of 12
  // heads of 64 to 1024: 8.8 us, 10.0 us in two spans).
  const int chunks = std::max(1, (a.H / a.G + 3) / 4);
  const int pairs = a.B * a.G * chunks, full = (L + 63) / 64;
  a.waves = pairs >= 256 ? 4 : 8;
  const int want = a.waves == 8 && L <= 65536 / D ? 1
      : std::max(1, std::min(full, (a.waves == 4 ? 512 : 256) / pairs));
  a.span = (full + want - 1) / want * 64;
  a.spans = (L + a.span - 1) / a.span;
  torch::Tensor part;
  a.part = nullptr;
  if (a.spans > 1) {
    part = torch::empty({(long)a.B * a.H * a.spans * (D + 2)},
                        qkv.options().dtype(torch::kFloat32));
    a.part = part.data_ptr<float>();
  }
  auto st = scaffold_stream();
  if (D == 32) launch<32>(a, st);
  else if (D == 64) launch<64>(a, st);
  else if (D == 128) launch<128>(a, st);
  else TORCH_CHECK(false, "decode_attention: head size ", D);
  HIP_CHECK(hipGetLastError());
  return out;
}
