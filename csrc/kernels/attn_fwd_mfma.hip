// K4 — MFMA flash attention forward (bf16, CDNA4 32x32x16).
//
// What bounds it: per 64 keys a wave of 32 query rows has 32 matrix
// instructions (heads of 128; 48 with weights in two parts) of 32 cycles, and
// some 1100 cycles of vector work: scale, maximum, exponential, sum and packing
// of 32 scores a lane.  One wave cannot do both at once, so a SIMD has two
// waves, of two blocks that nothing ties to each other: while one multiplies
// the other has its softmax.
//
//  * A block has 128 query rows, 4 waves of interleaved rows, so that all see
//    the same keys; Q stays in registers.
//  * A tile is S(t) = K(t) Q, O += V(t-1) P(t-1), softmax of S(t), one barrier.
//    K(t+1) and V(t) come into LDS meanwhile.  The four images are arrays of
//    their own: the compiler then knows that a read of one need not wait for
//    the copies into another.
//  * K image: rows with their 16-B chunks XORed; V image: units of 4 keys x 16
//    columns, for ds_read_b64_tr_b16.
//  * Swapped QK^T, so that softmax is lane-local, in base 2.
//
// In us, against one block of 8 waves with copies behind one another's waits:
// 2 x 32 x 4096 x 128 319 (860 TF/s) and 461, 16 x 12 x 1024 x 64 54 and 110, 1 x
// 32 x 512 x 128 17 and 28, 3 x 12 x 333 x 64 10.3 and 15.2; weights in two parts,
// 32 x 4096 x 128 202 and 337, 8 x 12 x 317 x 64 11.6 and 18.5, 32 x 1000 rows
// behind 2000 keys 88 and 144.  Those of the second kind as 8 waves in two groups
// that take turns by barriers 198, 15.9, 108; as blocks of 2 waves 291, 11.1, 104.
//
// Fragment maps verified on hardware by tests/ops/test_gpu_ops.py::
// test_mfma_layout_32x32x16 (probe.hip):
//   A(32x16): lane l -> row=l&31, k=8*(l>>5)+j
//   B(16x32): lane l -> col=l&31, k=8*(l>>5)+j
//   C(32x32): lane l, reg r -> col=l&31, row=(r&3)+8*(r>>2)+4*(l>>5)

#include "../common.h"

namespace {

constexpr int W = 4;               // waves of a block
constexpr int ROWS = 32 * W;       // query rows of a block

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short bf16x8_t __attribute__((ext_vector_type(8)));

DEVINL bf16x4 tr_at(const short* at) {
  typedef __attribute__((address_space(3))) bf16x4* P;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)at);
}

// the value of the lane 32 away
DEVINL float other_half(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, threadIdx.x & 32 ? r[0] : r[1]);
}

// S query rows see Sk keys, the last S of them their own places (training:
// S = Sk).  SPLIT: the weights enter the value product as two bf16 parts,
// hi + lo, 16 of float32's 24 significand bits (serving).  Against 64 bits the
// result is as near as with a float32 product, to five digits of its error
// (heads of 64 and 128, 2 to 4096 rows, up to 4096 keys): its own rounding to
// 8 bits is what there is.  An infinite value is infinite, or NaN where the weight's second
// part is none or of the other sign, in what sees it.
//
// KS = 2: the tiles of 64 keys go by turns to two groups of W waves, each with images of its
// own, and the first puts both results together at the end.
template <int D, bool SPLIT, int KS>
__global__ void __launch_bounds__(64 * W * KS, D == 64 && !SPLIT ? 4 : 2)
attn_fwd_mfma_kernel(const short* __restrict__ q, const short* __restrict__ k,
                   const short* __restrict__ v, short* __restrict__ o,
                   float* __restrict__ lse, int B, int H, int Hkv, int S,
                   int Sk, float scale2, int causal, int nbx, Strides4 qs,
                   Strides4 ks, Strides4 vs, Strides4 os) {
  constexpr int NSL = D / 16;
  constexpr int NDT = D / 32;
  constexpr int CH = D / 8;          // 16-B chunks per row
  constexpr int SLOTS = CH / W;      // of a wave, of an image
  static_assert(KS == 1 || SPLIT, "training's sums have an order");
  __shared__ __attribute__((aligned(16))) short k0s[KS * 64 * D], k1s[KS * 64 * D];
  __shared__ __attribute__((aligned(16))) short v0s[KS * 64 * D], v1s[KS * 64 * D];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wid = wave % W, group = KS > 1 ? wave / W : 0;
  short *const k0 = k0s + group * 64 * D, *const k1 = k1s + group * 64 * D;
  short *const v0 = v0s + group * 64 * D, *const v1 = v1s + group * 64 * D;
  const int l = threadIdx.x & 63;
  const int lq = l & 31;
  const int half = l >> 5;

  int bx, b, h;
  head_tile_map(nbx, B, H, Hkv, &bx, &b, &h);
  if (causal) bx = nbx - 1 - bx; // those that see most keys start first
  const int hk = h / (H / Hkv);
  // Rows of a wave: q0 + STEP * i + (its number).  Training: two blocks share 256
  // rows, again for the order of its sums, which of a wave's rows decide.
  constexpr int STEP = SPLIT ? W : 2 * W;
  const int q0 = (SPLIT ? bx : bx / 2) * 32 * STEP;
  if (q0 >= S) return;
  const int first = SPLIT ? wid : wid + W * (bx & 1);

  const long qb = (long)b * qs.sb + (long)h * qs.sh;
  const long kb = (long)b * ks.sb + (long)hk * ks.sh;
  const long vb = (long)b * vs.sb + (long)hk * vs.sh;

  const int qrow_g = q0 + STEP * lq + first;
  const int qrow = min(qrow_g, S - 1);
  const int off = Sk - S;            // place of the first row among the keys
  const short* qrow_ptr = q + qb + (long)qrow * qs.ss + 8 * half;
  bf16x8_t qf[NSL];
  #pragma unroll
  for (int s = 0; s < NSL; ++s) qf[s] = *(const bf16x8_t*)(qrow_ptr + 16 * s);

  f32x16_t oacc[NDT];
  #pragma unroll
  for (int t = 0; t < NDT; ++t) oacc[t] = {};
  // Training counts a score below -1e30 as masked.  Serving, whose scores no
  // loss keeps small, does not: an unseen key has -inf there, and every row
  // sees a key of the first tile, so that its maximum is a score from then on.
  constexpr float LOWEST = SPLIT ? -3.4028234663852886e38f : -1e30f;
  float m_run = LOWEST, l_run = 0.f;  // base-2 domain

  const int kv_end = causal ? min(Sk, off + q0 + 32 * STEP) : Sk;
  // tiles of a group, and of the first, which has the most: all meet at its barriers
  const int all = (kv_end + 63) / 64, most = (all + KS - 1) / KS;
  const int n = (all - group + KS - 1) / KS;

  // Copies of K(t) and V(t) into LDS, as buffer loads: what lies behind the last
  // key reads as zero, a lane's place in a tile is the same in every tile, and,
  // unlike global ones, they leave the count of LDS reads alone.
  unsigned ko[SLOTS], vo[SLOTS];
  auto order = [](int row) INLINE { return SPLIT ? swapped(row) : row; };
  #pragma unroll
  for (int it = 0; it < SLOTS; ++it) {
    const int s16 = (it * W + wid) * 64 + l;
    ko[it] = 2u * ((s16 / CH) * (unsigned)ks.ss + ((s16 % CH) ^ (order(s16 / CH) & 7)) * 8);
    const int sub = s16 / (4 * D), unit = s16 % (4 * D) >> 3, rem = s16 & 7;
    vo[it] = 2u * ((sub * 32 + 4 * (unit / (D / 16)) + (rem >> 1)) * (unsigned)vs.ss +
                   16 * (unit % (D / 16)) + 8 * (rem & 1));
  }
  auto copy = [&](short* to, const short* from, long ss, const unsigned* at, int t) INLINE {
    const long last = min(64, Sk - t * 64) - 1;
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(from + (long)t * 64 * ss), 0, (int)((last * ss + D) * 2), 0x00020000);
    #pragma unroll
    for (int it = 0; it < SLOTS; ++it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rows, (__attribute__((address_space(3))) void*)(to + (it * W + wid) * 512), 16,
          at[it], 0, 0, 0);
  };
  auto turn = []() INLINE {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // vmcnt(0), in a form that the compiler's own count takes notice of
  auto arrived = []() INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);
    asm volatile("" ::: "memory");
  };

  f32x16_t sacc[2];
  unsigned p[2][2][4], low[SPLIT ? 2 : 1][2][4];    // weights, [sub][16 keys]

  // Serving: rows of the score product are keys in swapped() order, so that lane
  // (lq, half) has, in registers 8 i ..., the weights of keys 16 i + 8 half ...,
  // which is what the value product takes from it.  Training: keys in order, and
  // the halves exchange their weights, because the sums then run over the keys
  // as they always have: through the layers of a model any other order of the
  // sums' roundings ends in gradients that differ as much as bf16 lets them.
  auto scores = [&](const short* kimg) INLINE {
    sacc[0] = {};
    sacc[1] = {};
    #pragma unroll
    for (int s = 0; s < NSL; ++s)
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int krow = sub * 32 + order(lq);
        const int chunk = (2 * s + half) ^ (lq & 7);
        const bf16x8_t kf = *(const bf16x8_t*)(kimg + krow * D + chunk * 8);
        sacc[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[s], sacc[sub], 0, 0, 0);
      }
  };
  const int tr = 64 * (lq >> 4) + ((l & 15) >> 2) * 16 + (l & 3) * 4 +
                 (half ? 128 * (D / 16) : 0);
  auto values = [&](const short* vimg) INLINE {
    auto frag = [&](int at) INLINE {
      return __builtin_shufflevector(tr_at(vimg + tr + at),
                                     tr_at(vimg + tr + at + 64 * (D / 16)),
                                     0, 1, 2, 3, 4, 5, 6, 7);
    };
    #pragma unroll
    for (int sub = 0; sub < 2; ++sub)
      #pragma unroll
      for (int t = 0; t < NDT; ++t)
        #pragma unroll
        for (int s = 0; s < 2; ++s) {
          const bf16x8_t vf = frag(sub * 32 * D + 64 * (4 * s * (D / 16) + 2 * t));
          oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              vf, *(const bf16x8_t*)p[sub][s], oacc[t], 0, 0, 0);
          if constexpr (SPLIT)
            oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                vf, *(const bf16x8_t*)low[sub][s], oacc[t], 0, 0, 0);
        }
  };
  auto softmax = [&](int c0) INLINE {
    if ((causal && c0 + 63 > q0 + first + off) || c0 + 64 > Sk) {
      const int end = (causal ? min(Sk, qrow_g + off + 1) : Sk) - c0 - (SPLIT ? 8 : 4) * half;
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          if (sub * 32 + (SPLIT ? 16 * (r >> 3) + (r & 7) : (r & 3) + 8 * (r >> 2)) >= end) sacc[sub][r] = -INFINITY;
    }
    #pragma unroll
    for (int sub = 0; sub < 2; ++sub)
      #pragma unroll
      for (int r = 0; r < 16; ++r) sacc[sub][r] *= scale2;
    float top = sacc[0][0];
    #pragma unroll
    for (int sub = 0; sub < 2; ++sub)
      #pragma unroll
      for (int r = 0; r < 16; ++r) top = fmaxf(top, sacc[sub][r]);
    float alpha = -1.f;                    // the maximum stays
    if (__any(top > m_run)) {
      top = fmaxf(top, other_half(top));
      const float m_new = fmaxf(m_run, top);
      alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      if constexpr (SPLIT) l_run *= alpha;
      #pragma unroll
      for (int t = 0; t < NDT; ++t)
        #pragma unroll
        for (int r = 0; r < 16; ++r) oacc[t][r] *= alpha;
    }
    float psum = 0.f;
    #pragma unroll
    for (int sub = 0; sub < 2; ++sub)
      #pragma unroll
      for (int s = 0; s < 2; ++s) {
        float e[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          e[j] = __builtin_amdgcn_exp2f(sacc[sub][8 * s + j] - m_run);
          psum += e[j];
        }
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned w = cvt_pk_bf16(e[2 * j], e[2 * j + 1]);
          p[sub][s][j] = w;
          if constexpr (SPLIT)
            low[sub][s][j] =
                cvt_pk_bf16(e[2 * j] - __builtin_bit_cast(float, w << 16),
                            e[2 * j + 1] - __builtin_bit_cast(float, w & 0xffff0000u));
        }
        if constexpr (!SPLIT) {
          unsigned(&w)[4] = p[sub][s];
          const auto rx = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
          const auto ry = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
          w[0] = rx[0];
          w[1] = ry[0];
          w[2] = rx[1];
          w[3] = ry[1];
        }
      }
    if constexpr (SPLIT) {
      l_run += psum;                       // of this lane's keys, until the end
    } else {
      const float other = other_half(psum);
      const float grown = fmaf(l_run, alpha, psum) + other, same = l_run + (psum + other);
      l_run = alpha < 0.f ? same : grown;
    }
  };
  // copies of a phase pair: K(u) and V(u - 1), for u up to n
  auto stage = [&](auto odd, int u) INLINE {
    if (u < n) copy(odd ? k1 : k0, k + kb, ks.ss, ko, KS * u + group);
    copy(odd ? v0 : v1, v + vb, vs.ss, vo, KS * (u - 1) + group);
  };
  auto tile = [&](auto odd, auto first, int t) INLINE {
    constexpr bool O = decltype(odd)::value;
    if (KS > 1 && t >= n) {
      turn();
      return;
    }
    stage(std::integral_constant<bool, !O>{}, t + 1);
    __builtin_amdgcn_s_setprio(1);
    scores(O ? k1 : k0);
    if constexpr (!decltype(first)::value) values(O ? v0 : v1);
    // operands come from LDS four ahead of the product that takes them
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    #pragma unroll
    for (int i = 0; i < 2 * NSL - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if constexpr (!decltype(first)::value) {
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      #pragma unroll
      for (int i = 0; i < 4 * NDT - 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, SPLIT ? 2 : 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    softmax((KS * t + group) * 64);
    arrived();
    turn();
  };
  constexpr std::true_type yes;
  constexpr std::false_type no;
  if (KS == 1 || n > 0) copy(k0, k + kb, ks.ss, ko, group);
  arrived();
  turn();
  tile(no, yes, 0);
  for (int t = 1; t < most; t += 2) {
    tile(yes, no, t);
    if (t + 1 < most) tile(no, no, t + 1);
  }
  if (n & 1) values(v0);
  else if (KS == 1 || n > 0) values(v1);
  if constexpr (SPLIT) l_run += other_half(l_run);

  if constexpr (KS == 2) {
    turn();                                // no image is read any more
    float *lo = (float*)k0s, *hi = (float*)k1s, *sums = (float*)v0s;
    const int at = wid * 64 + l;
    if (group) {
      #pragma unroll
      for (int t = 0; t < NDT; ++t)
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          (t < NDT / 2 ? lo : hi)[(t % (NDT / 2) * 16 + r) * 64 * W + at] = oacc[t][r];
      sums[at] = m_run;
      sums[64 * W + at] = l_run;
    }
    turn();
    if (group) return;
    const float m1 = sums[at], l1 = sums[64 * W + at], m = fmaxf(m_run, m1);
    const float f0 = __builtin_amdgcn_exp2f(m_run - m), f1 = __builtin_amdgcn_exp2f(m1 - m);
    m_run = m;
    l_run = l_run * f0 + l1 * f1;
    #pragma unroll
    for (int t = 0; t < NDT; ++t)
      #pragma unroll
      for (int r = 0; r < 16; ++r)
        oacc[t][r] = oacc[t][r] * f0 +
                     (t < NDT / 2 ? lo : hi)[(t % (NDT / 2) * 16 + r) * 64 * W + at] * f1;
  }

  // serving: -inf throughout is NaN, as in a softmax
  const float inv_l = SPLIT || l_run > 0.f ? 1.f / l_run : 0.f;
  if (qrow_g < S) {
    const long obase = (long)b * os.sb + (long)h * os.sh + (long)qrow_g * os.ss;
    // a lane has four consecutive columns in every four registers
    #pragma unroll
    for (int t = 0; t < NDT; ++t)
      #pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        bf16x4 pk;
        #pragma unroll
        for (int j = 0; j < 4; ++j) pk[j] = f2bf(oacc[t][rq * 4 + j] * inv_l);
        *(bf16x4*)(o + obase + 32 * t + 8 * rq + 4 * half) = pk;
      }
    if (half == 0 && lse)
      // lse contract is NATURAL log (backward consumes it):
      // max and sum ran in base 2, so lse = ln2 * (m2 + log2(l))
      lse[((long)b * H + h) * S + qrow_g] =
          0.6931471805599453f * (m_run + __log2f(fmaxf(l_run, 1e-30f)));
  }
}

}  // namespace

// A lane's place in a tile of 64 keys is a 32-bit offset: views whose keys lie
// farther apart than that allows are copied.
static torch::Tensor near_keys(const torch::Tensor& t) {
  return t.stride(2) < (1l << 24) ? t : t.contiguous();
}

template <int D, bool SPLIT>
static void launch(const torch::Tensor& q, const torch::Tensor& k,
                   const torch::Tensor& v, const torch::Tensor& o, float* lse,
                   int Sk, float scale2, bool causal, hipStream_t st) {
  const int B = (int)q.size(0), H = (int)q.size(1), S = (int)q.size(2);
  const int nbx = SPLIT ? (S + ROWS - 1) / ROWS : (S + 2 * ROWS - 1) / (2 * ROWS) * 2;
  auto kernel = attn_fwd_mfma_kernel<D, SPLIT, 1>;
  int waves = W;
  // Serving, blocks for no more than every unit: two groups of waves share the keys, so that
  // a SIMD has two waves that nothing ties to each other between barriers.  In us, one group and
  // two, heads of 64: 1 row of 12 heads x 1000 22.5 and 19.1, x 333 10.8 and 9.8, 4 x 12 x 600 16.9
  // and 15.1, 12 x 1000 rows behind 2000 keys 57 and 44, 10 x 12 x 256 behind 700 23.3 and 20.7; of
  // 128, 32 x 1000 32.3 and 28.8, 1000 rows behind 2000 84 and 74, 2 x 32 x 400 18.8 and 18.2.  Of
  // few keys what the groups save goes into their meeting: 32 x 300 x 128 12.7 and 13.3, 4 x 12 x 317
  // x 64 10.4 and 10.3.  With more blocks a unit has its two waves to a SIMD without: 8 x 12 x 317 x
  // 64 (288 blocks) 11.7 and 14.1, 32 x 1200 behind 2000 keys (320) 100 and 114; causal heads of 64
  // whose blocks differ most gain all the same (12 x 3000, 288, 56 and 45), 8 x 12 x 317 behind 700,
  // as many, do not (28 and 34).
  if constexpr (SPLIT) {
    if (Sk > 320 && (long)nbx * B * H <= 256) {
      kernel = attn_fwd_mfma_kernel<D, SPLIT, 2>;
      waves = 2 * W;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(nbx * B * H), dim3(64 * waves), 0,
                     st, (const short*)q.data_ptr(), (const short*)k.data_ptr(),
                     (const short*)v.data_ptr(), (short*)o.data_ptr(), lse, B, H,
                     (int)k.size(1), S, Sk, scale2, causal ? 1 : 0, nbx, strides_of(q),
                     strides_of(k), strides_of(v), strides_of(o));
}

void attn_fwd_mfma(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                   torch::Tensor o, torch::Tensor lse, double scale, bool causal) {
  // softmax runs in base 2
  const float scale2 = (float)scale * 1.4426950408889634f;
  const int D = (int)q.size(3), S = (int)q.size(2);
  k = near_keys(k);
  v = near_keys(v);
  auto st = scaffold_stream();
  if (D == 64) launch<64, false>(q, k, v, o, lse.data_ptr<float>(), S, scale2, causal, st);
  else if (D == 128) launch<128, false>(q, k, v, o, lse.data_ptr<float>(), S, scale2, causal, st);
  else TORCH_CHECK(false, "attn_fwd_mfma: unsupported D ", D);
  HIP_CHECK(hipGetLastError());
}

// Serving: causal attention of S rows behind Sk - S cached keys, weights as two
// bf16 parts.  q (B, H, S, D), k, v (B, Hkv, >= Sk, D), o (B, H, S, D)
// views with contiguous last dimensions.
void attn_prompt(const torch::Tensor& q, const torch::Tensor& k,
                 const torch::Tensor& v, const torch::Tensor& o, int Sk,
                 hipStream_t st) {
  const int D = (int)q.size(3);
  const float scale2 = 1.4426950408889634f / std::sqrt((float)D);
  const auto kn = near_keys(k), vn = near_keys(v);
  if (D == 64) launch<64, true>(q, kn, vn, o, nullptr, Sk, scale2, true, st);
  else if (D == 128) launch<128, true>(q, kn, vn, o, nullptr, Sk, scale2, true, st);
  else TORCH_CHECK(false, "attn_prompt: head size ", D);
}

torch::Tensor prompt_attention(torch::Tensor q, torch::Tensor k,
                               torch::Tensor v, long Sk) {
  CHECK_CUDA(q); CHECK_CUDA(k); CHECK_CUDA(v);
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes() &&
              k.size(0) == q.size(0) && k.size(3) == q.size(3) &&
              k.size(1) > 0 && q.size(1) % k.size(1) == 0 &&
              q.size(2) >= 1 && Sk >= q.size(2) && Sk <= k.size(2),
              "prompt_attention: shapes");
  for (const auto& t : {q, k, v})
    TORCH_CHECK(t.scalar_type() == torch::kBFloat16 && t.stride(3) == 1 &&
                t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
                t.stride(2) % 8 == 0 && (size_t)t.data_ptr() % 16 == 0,
                "prompt_attention: bf16, rows 16-byte aligned");
  auto o = torch::empty({q.size(0), q.size(2), q.size(1), q.size(3)},
                        q.options()).transpose(1, 2);
  attn_prompt(q, k, v, o, (int)Sk, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return o;
}
