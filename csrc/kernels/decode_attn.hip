// Decode attention over a dense key/value cache (bf16): one new token per
// row, every row at its own depth.
//
// One launch takes the packed projections [q heads | k heads | v heads] of
// the new tokens, turns q and k, appends k and v to the cache and attends:
// the block that owns the token's place puts the new key and value among the
// cached ones and stores them, the others read what is cached.
//
// What bounds it is reading the cache once.  A block has one kv head of one
// row and one span of the keys.  Spans exist so that few rows fill the chip;
// depths are read on the device, and blocks behind a row's depth end at once,
// so the grid is the same at every depth and a step can be captured.  Scores,
// softmax and sums are float32.

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
  int matrix;                    // decode_group_kernel
  int rows, eager;               // of a cache; decode_group_kernel
  long limit;                    // positions that exist: cache and tables
  float scale2;                  // of scores, times log2(e)
};

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

// column d of a head's sums over span s
template <int D>
DEVINL void put(const DecodeArgs& a, int b, int h, int s, int d, float top,
                float den, float num) {
  if (a.spans == 1) {
    a.out[((long)b * a.H + h) * D + d] = f2bf(num / den);
    return;
  }
  float* part = a.part + (((long)b * a.H + h) * a.spans + s) * (D + 2);
  part[d] = num;
  if (d == 0) {
    part[D] = top;
    part[D + 1] = den;
  }
}

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

// One or two query heads to a kv head.  A lane has 8 columns of a key, 16 lanes a
// key of 128; a cached row goes from memory to the registers that use it, and
// each group of lanes keeps a running maximum of its own until the end.
// D: head size; N: query heads of a block; WAVES: of a block
template <int D, int N, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
decode_head_kernel(DecodeArgs a) {
  constexpr int LPK = D / 8;            // lanes per key
  constexpr int KPI = 64 / LPK;         // keys per load of a wave
  constexpr int U = 4;                  // loads in flight
  constexpr int TILE = KPI * U;
  __shared__ float sm[WAVES][N][2], so[WAVES][N][D];

  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int g = l / LPK, c = l % LPK;   // key within a load, column chunk
  const int s = blockIdx.x, b = blockIdx.y / a.G, kv = blockIdx.y % a.G;
  const int h0 = kv * N;

  const long pos = a.pos[(long)b * a.pos_step];
  const bool on = (!a.active || a.active[b]) && pos >= 0 && pos < a.limit;
  const int lo = s * a.span;
  if (!on) {
    // nothing is written for the row; a place outside the cache shows
    if (s == 0 && w == 0)
      for (int i = l; i < N * D; i += 64)
        a.out[((long)b * a.H + h0) * D + i] = !a.active || a.active[b] ? 0x7fc0 : 0;
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
  float q[N][8], m[N], sum[N], o[N][8];
  #pragma unroll
  for (int r = 0; r < N; ++r) {
    const bf16x8 turn = turned<D>(a, row + (h0 + r) * D, c, p);
    m[r] = NONE;
    sum[r] = 0.f;
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
      q[r][i] = bf2f(turn[i]) * a.scale2;
      o[r][i] = 0.f;
    }
  }
  auto take = [&](const bf16x8 (&kk)[U], bf16x8 (&vv)[U], int j0) {
    // no weight makes an infinite value nothing, so those of the repeated
    // places go; only a row's last tile has some
    if (j0 + TILE > hi) {
      #pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u * KPI + g >= hi) vv[u] = bf16x8{};
    }
    float sc[U][N];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool see = j0 + u * KPI + g < hi;
      #pragma unroll
      for (int r = 0; r < N; ++r) {
        float d = 0.f;
        #pragma unroll
        for (int i = 0; i < 8; ++i) d = fmaf(q[r][i], bf2f(kk[u][i]), d);
        d = group_sum<LPK>(d);
        sc[u][r] = see ? d : NONE;
      }
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) {
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
    for (int u = 0; u < U; ++u)
      #pragma unroll
      for (int r = 0; r < N; ++r) {
        // a score of NONE is no key, also where the maximum is none yet
        const float e = sc[u][r] <= NONE ? 0.f : __builtin_amdgcn_exp2f(sc[u][r] - m[r]);
        sum[r] += e;
        #pragma unroll
        for (int i = 0; i < 8; ++i) o[r][i] = fmaf(e, bf2f(vv[u][i]), o[r][i]);
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
    if (g == 0) {
      *(bf16x8*)(kc + (long)p * a.ss) = nk;
      *(bf16x8*)(vc + (long)p * a.ss) = nv;
    } else {
      nv = bf16x8{};
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) {
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
  for (int r = 0; r < N; ++r) {
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
  for (int i = threadIdx.x; i < N * D; i += 64 * WAVES) {
    const int r = i / D, d = i % D;
    float t = NONE, den = 0.f, num = 0.f;
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) t = fmaxf(t, sm[x][r][0]);
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) {
      const float f = __builtin_amdgcn_exp2f(sm[x][r][0] - t);
      den += f * sm[x][r][1];
      num += f * so[x][r][d];
    }
    put<D>(a, b, h0 + r, s, d, t, den, num);
  }
}

DEVINL f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  typedef __attribute__((ext_vector_type(8))) __bf16 v8;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// Query heads that share keys, up to 8 of them in a block; a wave takes 32 keys
// at a time.  Keys go from memory to the registers that are the score product's
// operand, values through an LDS image of the wave's own, whose transpose reads
// make the value product's: no barrier in the loop, and the next tile's rows
// are on their way while one is used.  The 16 columns of a matrix instruction
// are 8 heads twice: the weights enter the value product as three bf16 parts, all
// of float32's bits, the second ones in the second 8 columns, the third ones by
// an instruction of their own (1 to 5 % of the time).  Of 64 rows, 32 heads of 128
// on 8, 1024 to 4096 keys deep, 671 MB: 128 us, 5.2 TB/s (148 with both products
// on the vector unit, which took half of the time there); one head to a kv head
// is left to it, 64 rows of 12 heads of 64 to 1024 keys 27.1 and 28.2 us, 1 row to
// 512 5.4 and 6.9, and two where decode_attention() says.
constexpr int R = 8;                    // query heads of a block
constexpr int WAVES = 4;                // of a block
constexpr int TILE = 32;                // keys of a wave at a time
// of a score, taken before the product: exact, and keeps its sums as far from
// the largest float as scaled queries would
constexpr float PRE = 0.125f;

// LDS of a wave: 32 rows of values, 16 of which lie in all banks, then the new
// key and value
template <int D> constexpr int row_of() { return D + 16; }
template <int D> constexpr int image_of() { return TILE * row_of<D>() + 2 * D; }

// D: head size
template <int D>
__global__ void __launch_bounds__(64 * WAVES, D == 128 ? 3 : 4)
decode_group_kernel(DecodeArgs a) {
  constexpr int NS = D / 32;            // steps of the score product
  constexpr int DT = D / 16;            // tiles of 16 columns
  constexpr int LPK = D / 8;            // lanes per value row
  constexpr int KPI = 64 / LPK;         // value rows per load of a wave
  constexpr int NV = TILE / KPI;
  constexpr int ROW = row_of<D>();
  constexpr int MERGE = R * (D + 2) * 2;             // a wave's sums, shorts
  constexpr int IMAGE = image_of<D>() > MERGE ? image_of<D>() : MERGE;
  __shared__ __attribute__((aligned(16))) short lds[WAVES * IMAGE];

  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int lr = l & 15, lg = l >> 4;
  const int rep = a.H / a.G, chunks = (rep + R - 1) / R;
  const int s = blockIdx.x;
  const int b = blockIdx.y / (a.G * chunks);
  const int kv = blockIdx.y / chunks % a.G, ch = blockIdx.y % chunks;
  const int h0 = kv * rep + ch * R, heads = min(R, rep - ch * R);

  short* kc = a.k + b * a.sb + kv * a.sh;
  short* vc = a.v + b * a.sb + kv * a.sh;
  short* image = lds + w * IMAGE;
  short* fresh = image + TILE * ROW;        // new key, new value

  // Keys: lane (lg, lr) has columns 32 s + 8 lg of key lr, as the operand of
  // the product wants them.  Values: whole rows.  Places behind the last key
  // repeat it and do not count; the new token's place has not been written.
  // Where blocks are few the first tile is asked for before the depth is known.
  const int lo = s * a.span;
  int j = lo + w * TILE, last = a.rows - 1;
  bf16x8 kk[2][NS], vv[NV];
  auto fetch_k = [&](int j0) {
    #pragma unroll
    for (int t = 0; t < 2; ++t) {
      const short* at = kc + (long)min(j0 + 16 * t + lr, last) * a.ss + 8 * lg;
      #pragma unroll
      for (int n = 0; n < NS; ++n) kk[t][n] = *(const bf16x8*)(at + 32 * n);
    }
  };
  auto fetch_v = [&](int j0) {
    #pragma unroll
    for (int n = 0; n < NV; ++n)
      vv[n] = *(const bf16x8*)(
          vc + (long)min(j0 + n * KPI + l / LPK, last) * a.ss + 8 * (l % LPK));
  };
  if (a.eager) {
    fetch_k(j);
    fetch_v(j);
  }

  const long pos = a.pos[(long)b * a.pos_step];
  const bool on = (!a.active || a.active[b]) && pos >= 0 && pos < a.limit;
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
  const int hi = min(p + 1, lo + a.span);   // keys [lo, hi)
  const bool own = p < hi;                  // the new key is one of them
  last = hi - 1;
  if (!a.eager && j < hi) {
    fetch_k(j);
    fetch_v(j);
  }
  const short* row = a.qkv + (long)b * a.ldq;
  if (own && l < LPK) {
    const bf16x8 nk = turned<D>(a, row + (a.H + kv) * D, l, p);
    const bf16x8 nv = *(const bf16x8*)(row + (a.H + a.G + kv) * D + 8 * l);
    *(bf16x8*)(fresh + 8 * l) = nk;
    *(bf16x8*)(fresh + D + 8 * l) = nv;
    if (w == 0 && ch == 0) {
      *(bf16x8*)(kc + (long)p * a.ss + 8 * l) = nk;
      *(bf16x8*)(vc + (long)p * a.ss + 8 * l) = nv;
    }
  }
  bf16x8 q[NS];
  #pragma unroll
  for (int n = 0; n < NS; ++n) {
    q[n] = turned<D>(a, row + (h0 + min(lr & (R - 1), heads - 1)) * D, 4 * n + lg, p);
    #pragma unroll
    for (int i = 0; i < 8; ++i) q[n][i] = f2bf(bf2f(q[n][i]) * PRE);
  }
  const float scale = a.scale2 / PRE;
  float m = NONE, sum = 0.f;                // of head lr, of the lane's keys
  f32x4 o[DT];
  #pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a transpose read of 4 rows x 16 columns: rows 4 lg ...
  const unsigned tr = lds_byte_off(image) +
                      ((4 * lg + (lr >> 2)) * ROW + (lr & 3) * 4) * 2;

  for (; j < hi; j += WAVES * TILE) {
    const int next = j + WAVES * TILE;
    if (j + TILE >= hi) {
      // the last tile: the new token comes in, and what is behind it goes: no
      // weight makes an infinite value nothing
      #pragma unroll
      for (int t = 0; t < 2; ++t)
        if (own && j + 16 * t + lr == p)
          #pragma unroll
          for (int n = 0; n < NS; ++n)
            kk[t][n] = *(const bf16x8*)(fresh + 32 * n + 8 * lg);
      #pragma unroll
      for (int n = 0; n < NV; ++n) {
        const int at = j + n * KPI + l / LPK;
        if (own && at == p) vv[n] = *(const bf16x8*)(fresh + D + 8 * (l % LPK));
        if (at >= hi) vv[n] = bf16x8{};
      }
    }
    #pragma unroll
    for (int n = 0; n < NV; ++n)
      *(bf16x8*)(image + (n * KPI + l / LPK) * ROW + 8 * (l % LPK)) = vv[n];
    if (next < hi) fetch_v(next);
    f32x4 sc[2];
    #pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      #pragma unroll
      for (int n = 0; n < NS; ++n) sc[t] = mma(kk[t][n], q[n], sc[t]);
    }
    if (next < hi) fetch_k(next);
    float top = NONE;
    #pragma unroll
    for (int t = 0; t < 2; ++t)
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[t][r] *= scale;
        if (j + TILE > hi && j + 16 * t + 4 * lg + r >= hi) sc[t][r] = -INFINITY;
        top = fmaxf(top, sc[t][r]);
      }
    if (__any(top > m)) {
      top = fmaxf(top, __shfl_xor(top, 16, 64));
      top = fmaxf(fmaxf(top, __shfl_xor(top, 32, 64)), m);
      const float f = __builtin_amdgcn_exp2f(m - top);
      m = top;
      sum *= f;
      #pragma unroll
      for (int t = 0; t < DT; ++t) o[t] *= f;
    }
    // weights of the keys 16 t + 4 lg + r; the value product's sum runs over
    // the keys in this order
    bf16x8 e, f;
    float part = 0.f;
    #pragma unroll
    for (int t = 0; t < 2; ++t)
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = __builtin_amdgcn_exp2f(sc[t][r] - m);
        part += x;
        const WeightParts c = weight_parts(x);
        e[4 * t + r] = lr < R ? c.hi : c.mid;
        // next to nothing in the columns that have no third part
        f[4 * t + r] = lr < R ? c.lo : x > 0.f ? 0x0080 : 0;
      }
    sum += part;
    #pragma unroll
    for (int t = 0; t < DT; ++t) {
      const bf16x8 v = tr_read_frag(tr + 32 * t, tr + 32 * t + 16 * ROW * 2);
      o[t] = mma(v, e, o[t]);
      o[t] = mma(v, f, o[t]);
    }
  }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  // the parts, then waves
  float* mine = (float*)image;              // [R][D + 2]
  #pragma unroll
  for (int t = 0; t < DT; ++t) {
    #pragma unroll
    for (int i = 0; i < 4; ++i) o[t][i] += __shfl_xor(o[t][i], R, 64);
    if (lr < heads)
      #pragma unroll
      for (int i = 0; i < 4; ++i) mine[lr * (D + 2) + 16 * t + 4 * lg + i] = o[t][i];
  }
  if (l < heads) {
    mine[l * (D + 2) + D] = m;
    mine[l * (D + 2) + D + 1] = sum;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < heads * D; i += 64 * WAVES) {
    const int r = i / D, d = i % D, h = h0 + r;
    const float* of = (const float*)lds + r * (D + 2);
    float t = NONE, den = 0.f, num = 0.f;
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) t = fmaxf(t, of[x * (IMAGE / 2) + D]);
    #pragma unroll
    for (int x = 0; x < WAVES; ++x) {
      const float* from = of + x * (IMAGE / 2);
      const float f = __builtin_amdgcn_exp2f(from[D] - t);
      den += f * from[D + 1];
      num += f * from[d];
    }
    put<D>(a, b, h, s, d, t, den, num);
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

template <int D, int N>
void launch_heads(const DecodeArgs& a, hipStream_t st) {
  const dim3 grid(a.spans, a.B * a.G);
  if (a.waves == 8)
    hipLaunchKernelGGL((decode_head_kernel<D, N, 8>), grid, dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((decode_head_kernel<D, N, 4>), grid, dim3(256), 0, st, a);
}

template <int D>
void launch(const DecodeArgs& a, hipStream_t st) {
  if (a.matrix) {
    const int chunks = (a.H / a.G + R - 1) / R;
    hipLaunchKernelGGL((decode_group_kernel<D>), dim3(a.spans, a.B * a.G * chunks),
                       dim3(64 * WAVES), 0, st, a);
  } else if (a.H == a.G) {
    launch_heads<D, 1>(a, st);
  } else {
    launch_heads<D, 2>(a, st);
  }
  if (a.spans > 1)
    hipLaunchKernelGGL((decode_merge_kernel<D>), dim3(a.B * a.H),
                       dim3(D < 64 ? 64 : D), 0, st, a);
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
  TORCH_CHECK(L > 0, "decode_attention: a cache without places");
  const int rep = a.H / a.G, chunks = (rep + R - 1) / R;
  const int pairs = a.B * a.G * chunks, full = (L + 63) / 64;
  // Two heads to a kv head use a quarter of the matrix instruction's columns, and
  // the vector kernel's 8 waves walk a span faster than the other's 4; in us,
  // vector and matrix kernel: heads of 128, 64 pairs of a row and a kv head, caches
  // of 128 5.7 and 6.7, 1024 10.5 and 11.5, 512 pairs of 128 7.3 and 9.3; heads of
  // 64, 64 pairs of 128 5.6 and 5.1, of 1024 9.5 and 10.6; heads of 32, 64 pairs of
  // 128 5.4 and 4.4, of 1024 7.4 and 9.1, 512 of 4096 32.1 and 32.8.  The matrix
  // kernel's where it starts sooner, or its products are what counts: heads of
  // 128, 256 pairs of 1024 21.6 and 19.5, 512 of 4096 130 and 125; of 64, 256 of 1024
  // 15.1 and 11.7.
  if (rep == 2)
    a.matrix = D == 128 ? L > 256 && pairs >= 192 && (long)pairs * L >= 128 * 1024
                        : L <= 256 || (D == 64 && pairs >= 256);
  else
    a.matrix = rep > 2;
  // Spans of whole 64s.  Vector kernel: with 256 pairs or more, 512 blocks of 4
  // waves fill the chip (64 rows of 12 heads of 64 to 1024 deep: 27 us); with
  // fewer, 256 blocks of 8 waves.  A cache that 8 waves walk in 4 steps is one
  // span, which saves the merge (8 rows of 12 heads of 64 to 1024: 8.8 us, 10.0 us
  // in two spans); of two heads, what 4 waves do as well (32 rows of 8 pairs of
  // 128, 128 deep: 6.0 and 8.8).
  // Matrix kernel: a compute unit's misses bound it to 50 KB a microsecond (what
  // 32 keys cost aside, which rows of 32 do not come below), so up to 256 blocks
  // share the keys, if that saves more than the merge's 5 us; in us, one span and
  // several: 1 row of 8 kv heads to 4096 43 and 16, 4 rows to 1000 17.3 and 13.0, 8
  // rows to 2048 30 and 21, 16 rows to 1000 19.9 and 19.3, 32 rows to 300 13.7 and
  // 18.0; 4 heads of 32, 16 rows to 4096 24.8 and 18.7.
  int want;
  if (a.matrix) {
    want = std::max(1, std::min((full + 1) / 2, 256 / pairs));
    if (4l * L * std::max(D, 64) * (want - 1) <= 256l * 1024 * want) want = 1;
    // A few more blocks than compute units leave some with two and most with one; three
    // spans a row share them out.  One span and three, us: 32 heads of 128 on 8, caches
    // of 4096 near their end, 33 rows 98 and 75, 40 104 and 87, 44 109 and 95, 48 111
    // and 107; while only 512 places are taken, 15.2 and 17.5, 15.9 and 19.6, 16.2 and
    // 21.3.  Caches of 2048 gain less than their first steps would lose (40 rows: 58
    // and 51), and so do heads of 64 (40 rows of 4096: 53 and 52).
    if (pairs > 256 && pairs <= 352 && (long)L * D >= 512l * 1024) want = 3;
  } else {
    a.waves = pairs >= 256 ? 4 : 8;
    want = std::max(1, std::min(rep == 1 ? full : (full + 1) / 2,
                                (a.waves == 4 ? 512 : 256) / pairs));
    if ((a.waves == 8 && L <= 65536 / D) || (rep == 2 && L <= 32768 / D)) want = 1;
  }
  a.span = (full + want - 1) / want * 64;
  a.spans = (L + a.span - 1) / a.span;
  a.rows = L;
  a.eager = (long)pairs * a.spans <= 512;
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
