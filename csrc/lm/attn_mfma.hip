// The bf16 prompt-attention kernels for head sizes that are multiples of 8
// up to 128 (attn.hip serves every other size and float32).
//
// A block owns one tile of up to 64 prompt rows for HPB query heads of one
// kv head; each head's rows are two waves of 32.  All 2*HPB waves share the
// staged page, so grouped heads pay for keys and values once.
//
//  * S^T = K Q^T with 32x32x16 MFMAs: a lane holds one query's scores for
//    32 of the page's 64 keys, so the softmax needs one cross-lane step.
//  * Pages are staged a page ahead, one barrier a page: by copies into LDS (as
//    stored), or through registers into the other half of a double buffer.
//    Keys past the tile's last token are staged as zeros (their cells may hold
//    anything).
//  * O^T = V^T P^T with V read through the LDS transpose reads.  P goes in
//    as two bf16 parts (hi + lo), so the weights keep 16 significand bits;
//    both parts share the V fragments.
//  * Tied form (values are keys): one image of a page serves both products,
//    rows for the scores, transpose reads for the values; the swizzle keeps
//    both free of conflicts.  A key's factor and its distance bias join the
//    score in one multiply-add each.
//  * Window form: soft cap by one exponential and one reciprocal, the bias by
//    distance from LDS (a page whose every distance is beyond the table's
//    last adds a constant), kept first pages before the window's.
//  * Tied and window forms: pages that no row of a wave sees are skipped by that
//    wave.  Masks are applied only on pages that a chunk edge or the diagonal crosses.

#include "lm.h"
#include "tile.h"
#include "attn.h"

namespace {

constexpr float LOG2E = 1.4426950408889634f;

DEVINL f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, a),
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, b), c, 0,
      0, 0);
}

// B fragments (16 keys each) of 16 consecutive-by-lane P^T values, which p
// holds afterwards less what went into them
DEVINL void p_frags(float (&p)[16], bf16x8 (&out)[2]) {
  #pragma unroll
  for (int s = 0; s < 2; ++s) {
    unsigned w[4];
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      float &x = p[8 * s + 2 * j], &y = p[8 * s + 2 * j + 1];
      w[j] = cvt_pk_bf16(x, y);
      x -= __builtin_bit_cast(float, w[j] << 16);
      y -= __builtin_bit_cast(float, w[j] & 0xffff0000u);
    }
    auto rx = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    auto ry = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    union { unsigned u[4]; bf16x8 v; } f;
    f.u[0] = rx[0]; f.u[1] = ry[0]; f.u[2] = rx[1]; f.u[3] = ry[1];
    out[s] = f.v;
  }
}

// f(this lane's, that of the lane 32 away)
template <typename F>
DEVINL float over_halves(float x, F f) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return f(__builtin_bit_cast(float, (unsigned)r[0]),
           __builtin_bit_cast(float, (unsigned)r[1]));
}

// this lane's columns of a row, times inv and, if there is a gate, its sigmoid
template <int NDT>
DEVINL void store_row(const AttnArgs& a, const f32x16 (&o)[NDT], float inv,
                      int row, int h, int half) {
  short* dst = (short*)a.out + (long)row * a.ldo + (long)h * a.vdim;
  const short* gate = a.gate ? (const short*)a.gate + (long)row * a.ld +
                                   (long)h * a.vdim : nullptr;
  #pragma unroll
  for (int i = 0; i < NDT; ++i)
    #pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int d = 32 * i + 8 * rq + 4 * half;
      if (d >= a.vdim) continue;
      bf16x4 pk, gt{};
      if (gate) gt = *(const bf16x4*)(gate + d);
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float y = o[i][rq * 4 + j] * inv;
        pk[j] = cvt_bf16(gate ? y * sigmoid(bf2f(gt[j])) : y);
      }
      *(bf16x4*)(dst + d) = pk;
    }
}

// Place of 8-column chunk cb of key j in a page's image.
template <int DK, bool TIED>
DEVINL int chunk_at(int j, int cb) {
  if constexpr (TIED) return tied_chunk<DK>(j, cb);
  else return cb ^ (j & 7);
}

constexpr int BIAS_LDS = 512;          // entries of a head's bias kept in LDS

// Tied, with a bias by distance, or else window
template <int DK, int DV, int HPB, bool TIED>
__global__ void __launch_bounds__(HPB * 128, 2)
attn_prefill_form_kernel(AttnArgs a, const int4* __restrict__ tiles,
                         int n_tiles) {
  constexpr int NT = HPB * 128;
  constexpr int NSL = DK / 16, NDT = DV / 32;
  constexpr bool BIAS = TIED, WIN = !TIED;
  static_assert(!TIED || DK == DV, "one image");
  constexpr int BUF = 64 * (DK + (TIED ? 0 : DV));  // K image + V tr-image
  constexpr int KC = 64 * DK / 8 / NT, VC = 64 * DV / 8 / NT;
  __shared__ __attribute__((aligned(16))) short lds[2 * BUF];
  __shared__ __attribute__((aligned(16))) float kfs[TIED ? 2 * 64 : 4];
  __shared__ float bias_s[WIN ? HPB * BIAS_LDS : 1];

  const int tid = threadIdx.x, l = tid & 63, wid = tid >> 6;
  const int lq = l & 31, half = l >> 5;
  int bx, by;
  xcd_tile_map(n_tiles, &bx, &by);
  bx = n_tiles - 1 - bx;               // a prompt's last tiles see most: first
  const int hg = a.H / a.G, nhc = hg / HPB;
  const int g = by / nhc;
  const int h = g * hg + (by % nhc) * HPB + (wid >> 1);
  const int4 t = tiles[bx];                    // first row, rows, pos0, slot
  const int row = 32 * (wid & 1) + lq;
  const int rowc = min(row, t.y - 1);
  const int ip = t.z + rowc;
  const int cs = first_seen(a, ip), keep = WIN ? a.keep : 0;

  bf16x8 qf[NSL];
  {
    const short* q = (const short*)a.qkv + (long)(t.x + rowc) * a.ld + (long)h * a.dim;
    #pragma unroll
    for (int s = 0; s < NSL; ++s) {
      const int c = 16 * s + 8 * half;
      qf[s] = c < a.dim ? *(const bf16x8*)(q + c) : bf16x8{};
    }
  }

  const int p_last = t.z + t.y - 1;
  const PageList pages(a, t.z, p_last);
  const int* tab = a.table + (long)t.w * a.max_pages;

  // this wave's rows: first and last position, and their chunk starts
  const int w0 = t.z + min(32 * (wid & 1), t.y - 1);
  const int w1 = t.z + min(32 * (wid & 1) + 31, t.y - 1);
  const bool w_any = 32 * (wid & 1) < t.y;
  const int wcs0 = first_seen(a, w0), wcs1 = first_seen(a, w1);

  bf16x8 kr[KC], vr[TIED ? 1 : VC];
  float kf = 0.f;
  const float scale2 = a.scale * LOG2E;
  auto stage_load = [&](int pg, long page) {
    const short* kp = (const short*)a.kc + (page * a.G + g) * LM_PAGE * a.dim;
    const int left = p_last - pg * LM_PAGE;    // last valid key of the page
    #pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int s = i * NT + tid, j = s / (DK / 8), c = (s % (DK / 8)) * 8;
      kr[i] = c < a.dim && (!TIED || j <= left)
                  ? *(const bf16x8*)(kp + (long)j * a.dim + c) : bf16x8{};
    }
    if constexpr (TIED) {
      if (tid < 64) kf = tid <= left ? a.ks[page * LM_PAGE + tid] * scale2 : 0.f;
    } else {
      const short* vp = (const short*)a.vc + (page * a.G + g) * LM_PAGE * a.vdim;
      #pragma unroll
      for (int i = 0; i < VC; ++i) {
        const int s = i * NT + tid, j = s / (DV / 8), c = (s % (DV / 8)) * 8;
        vr[i] = c < a.vdim && j <= left
                    ? *(const bf16x8*)(vp + (long)j * a.vdim + c) : bf16x8{};
      }
    }
  };
  auto stage_write = [&](int buf) {
    short* kd = lds + buf * BUF;
    short* vd = kd + 64 * DK;
    #pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int s = i * NT + tid, j = s / (DK / 8), cb = s % (DK / 8);
      *(bf16x8*)(kd + j * DK + chunk_at<DK, TIED>(j, cb) * 8) = kr[i];
    }
    if constexpr (TIED) {
      if (tid < 64) kfs[buf * 64 + tid] = kf;
    } else {
      #pragma unroll
      for (int i = 0; i < VC; ++i) {
        const int s = i * NT + tid, j = s / (DV / 8), c = (s % (DV / 8)) * 8;
        *(bf16x8*)(vd + ((j >> 2) * (DV / 16) + (c >> 4)) * 64 + (j & 3) * 16 +
                   (c & 15)) = vr[i];
      }
    }
  };
  // transpose reads: this lane's 8 bytes of a 4-key x 16-column subtile
  const unsigned tr0 = lds_byte_off(lds + 64 * DK) + 128u * (lq >> 4) +
                       ((l & 15) >> 2) * 32 + (l & 3) * 8 +
                       (half ? 128u * 2 * (DV / 16) : 0);
  // the same out of the tied image: row 8 * half + r of a 16-key step,
  // r = 0..3, and the chunk that chunk_at gives for it; steps, quads and
  // column tiles only flip bits of the chunk
  const int tr_r = (l & 15) >> 2;
  const unsigned tk0 = lds_byte_off(lds) + (8 * half + tr_r) * (DK * 2) + (l & 1) * 8;
  const unsigned tkc = chunk_at<DK, true>(8 * half + tr_r,
                                          2 * (lq >> 4) + ((l & 3) >> 1)) * 16;

  const float slope2 = BIAS && a.slopes ? a.slopes[h] * LOG2E : 0.f;
  float m_run = a.has_sink ? sink_score<false>(a, h) * LOG2E : -1e30f;
  float l_run = a.has_sink && !half ? 1.f : 0.f;    // of this half's keys
  f32x16 o[NDT];
  #pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = {};

  // window form: this head's bias in base 2
  const int n_bias = WIN ? a.n_bias : 0;
  const bool bias_lds = n_bias <= BIAS_LDS;
  const float* bias_g = nullptr;
  const float* bias_h = bias_s + (wid >> 1) * BIAS_LDS;
  float bias_far = 0.f;
  if constexpr (WIN) {
    bias_g = a.bias + (long)h * n_bias;
    bias_far = bias_g[n_bias - 1] * LOG2E;
    if (bias_lds)
      for (int i = tid % 128; i < n_bias; i += 128)
        bias_s[(wid >> 1) * BIAS_LDS + i] = bias_g[i] * LOG2E;
  }
  const SoftCap cap(a, LOG2E);

  stage_load(pages[0], tab[pages[0]]);
  stage_write(0);
  __syncthreads();
  int cur = 0;
  long next = tab[pages[min(1, pages.n - 1)]];   // a page's place, one early
  for (int it = 0; it < pages.n; ++it) {
    const int pg = pages[it];
    if (it + 1 < pages.n) stage_load(pages[it + 1], next);
    next = tab[pages[min(it + 2, pages.n - 1)]];
    const int j0 = pg * LM_PAGE;
    if (w_any && j0 <= w1 && (j0 + LM_PAGE > wcs0 || j0 < keep)) {
      const short* kimg = lds + cur * BUF;
      f32x16 s[2];
      s[0] = {};
      s[1] = {};
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int kr_ = sub * 32 + lq;
        #pragma unroll
        for (int i = 0; i < NSL; ++i)
          s[sub] = mma32(*(const bf16x8*)(kimg + kr_ * DK +
                                          chunk_at<DK, TIED>(kr_, 2 * i + half) * 8),
                         qf[i], s[sub]);
      }
      const bool edge = j0 + LM_PAGE - 1 > w0 || j0 < wcs1;
      float mt = -1e30f;
      const float d0 = slope2 * (float)(j0 + 4 * half - ip);
      if constexpr (WIN) {
        const int last = n_bias - 1, dist = ip - j0 - 4 * half;
        const bool far = w0 - j0 - (LM_PAGE - 1) >= last;     // of all rows
        float most = 0.f;
        #pragma unroll
        for (int sub = 0; sub < 2; ++sub)
          #pragma unroll
          for (int r = 0; r < 16; ++r) most = fmaxf(most, fabsf(s[sub][r]));
        const bool small = cap.small(most);
        // both are uniform in the wave
        auto scores = [&](auto bias) {
          #pragma unroll
          for (int sub = 0; sub < 2; ++sub)
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float b = bias(sub * 32 + (r & 3) + 8 * (r >> 2));
              s[sub][r] = small ? cap.near(s[sub][r], b) : cap.any(s[sub][r], b);
            }
        };
        if (far) {
          if (small) {
            #pragma unroll
            for (int sub = 0; sub < 2; ++sub)
              #pragma unroll
              for (int r = 0; r < 16; ++r) s[sub][r] = cap.near(s[sub][r], bias_far);
          } else {
            #pragma unroll
            for (int sub = 0; sub < 2; ++sub)
              #pragma unroll
              for (int r = 0; r < 16; ++r) s[sub][r] = cap.any(s[sub][r], bias_far);
          }
        } else if (bias_lds) {
          scores([&](int j) { return bias_h[min(max(dist - j, 0), last)]; });
        } else {
          scores([&](int j) { return bias_g[min(max(dist - j, 0), last)] * LOG2E; });
        }
      }
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int jr = sub * 32 + (r & 3) + 8 * (r >> 2);
          float x = s[sub][r];
          if constexpr (TIED) x *= kfs[cur * 64 + jr + 4 * half];
          else if constexpr (!WIN) x *= scale2;
          if constexpr (BIAS) x += fmaf(slope2, (float)jr, d0);
          if (edge) {
            const int j = j0 + jr + 4 * half;
            x = j <= ip && (j >= cs || (WIN && j < keep)) ? x : -1e30f;
          }
          s[sub][r] = x;
          mt = fmaxf(mt, x);
        }
      mt = over_halves(mt, [](float a, float b) { return fmaxf(a, b); });
      // a row that has seen no key of its own yet collects finite junk
      // here; its first own key sets m_run and wipes it (alpha = 0)
      if (__any(mt > m_run)) {
        const float mn = fmaxf(m_run, mt);
        const float al = __builtin_amdgcn_exp2f(m_run - mn);
        m_run = mn;
        l_run *= al;
        #pragma unroll
        for (int i = 0; i < NDT; ++i)
          #pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= al;
      }
      float ps = 0.f;
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[sub][r] = __builtin_amdgcn_exp2f(s[sub][r] - m_run);
          ps += s[sub][r];
        }
      l_run += ps;

      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        float p[16];
        #pragma unroll
        for (int r = 0; r < 16; ++r) p[r] = s[sub][r];
        bf16x8 hi[2], lo[2];
        p_frags(p, hi);
        p_frags(p, lo);
        const unsigned base = tr0 + (unsigned)cur * (BUF * 2) + (unsigned)sub * (32u * DV * 2);
        #pragma unroll
        for (int t2 = 0; t2 < NDT; t2 += 2) {
          auto addr = [&](int tt, int ss) {
            return base + 128u * (unsigned)((4 * ss) * (DV / 16) + 2 * tt);
          };
          const unsigned qs = 128u * (DV / 16);
          // column tile tt, 16-key step ss, quad q of it (tied image)
          auto tied = [&](int tt, int ss, int q) {
            const unsigned flip = (DK == 64 ? q : 8 * q) ^ (4 * tt);
            return tk0 + (unsigned)cur * (BUF * 2) +
                   (unsigned)(32 * sub + 16 * ss + 4 * q) * (DK * 2) +
                   (tkc ^ (flip * 16));
          };
          bf16x8_quad v;
          if constexpr (TIED)
            v = tr_read_quad(tied(t2, 0, 0), tied(t2, 0, 1), tied(t2, 1, 0),
                             tied(t2, 1, 1), tied(t2 + 1, 0, 0),
                             tied(t2 + 1, 0, 1), tied(t2 + 1, 1, 0),
                             tied(t2 + 1, 1, 1));
          else
            v = tr_read_quad(
              addr(t2, 0), addr(t2, 0) + qs, addr(t2, 1), addr(t2, 1) + qs,
              addr(t2 + 1, 0), addr(t2 + 1, 0) + qs, addr(t2 + 1, 1),
              addr(t2 + 1, 1) + qs);
          o[t2] = mma32(v.f[0], hi[0], o[t2]);
          o[t2 + 1] = mma32(v.f[2], hi[0], o[t2 + 1]);
          o[t2] = mma32(v.f[1], hi[1], o[t2]);
          o[t2 + 1] = mma32(v.f[3], hi[1], o[t2 + 1]);
          o[t2] = mma32(v.f[0], lo[0], o[t2]);
          o[t2 + 1] = mma32(v.f[2], lo[0], o[t2 + 1]);
          o[t2] = mma32(v.f[1], lo[1], o[t2]);
          o[t2 + 1] = mma32(v.f[3], lo[1], o[t2 + 1]);
        }
      }
    }
    // the other buffer's readers passed the barrier of the last page
    if (it + 1 < pages.n) stage_write(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }

  l_run = over_halves(l_run, [](float a, float b) { return a + b; });
  if (row < t.y) {
    const float inv = l_run > 0.f ? a.out_scale / l_run : 0.f;
    store_row<NDT>(a, o, inv, t.x + row, h, half);
  }
}

// As stored, with or without a bias by distance.  A page is S = K(t) Q, O += V(t
// - 1) P(t - 1), softmax of S, one barrier; K(t + 1) and V(t) come into LDS
// meanwhile, by buffer loads, which read as zero what lies behind the tile's
// last token or a head's columns.  The four images are arrays of their own: the
// compiler then knows that a read of one need not wait for copies into another.
// Rows of the score product are keys in swapped() order, so that a lane has the
// weights that the value product takes from it.  An unseen key has -inf.
//
// Bound by vector work beside 48 matrix instructions a page, and by a block's
// first loads, each behind another: 16 heads of 128 on 4, 8192 tokens in chunks
// of 1024 (8.5 pages a block) 92 us, against 119 with pages through registers
// and values behind their own page's softmax; two prompts of 1000 behind 1500
// 48 against 60.  Blocks of one head as well: 9 heads of 64 on 3 with values of 128,
// 8192 tokens in chunks of 1024, 95 against 121, 3 heads of 64 on 1 39 against 50, 5
// heads of 128 97 against 129; bounds that ask for more waves than LDS has room for
// are not kept, and 277 registers leave one wave to a SIMD (131, 43, 96).
//
// KS = 2, where blocks are no more than compute units: a page's keys are split over two
// waves of a SIMD, which add their results up at the end, for one wave alone has 8 cycles
// an instruction and waits between products and softmax.  Two prompts of 1000 behind 1500,
// 256 blocks, 47.6 -> 41.3 us.  (There, copies two pages ahead into three images take 51.)
// Of few pages the adding up is more than that saves.  In us, KS = 1 and 2: two heads a
// block, 16 of 128 on 4, 8 x 64 tokens (a page) 9.9 and 11.1, 4 x 128 (two) 11.8 and 13.0, 192
// (three) 13.6-14.6 and 14.0-14.2, 2 x 193 14.0-15.3 and 14.4-14.6, 300 (five) 17.6 and 16.3-16.9;
// of 64, 7.2 and 7.8, 8.6 and 8.7, 9.7 and 9.9, 10.6 and 10.5; one head, 8 of 128 9.8 and 10.1,
// 11.9 and 11.6, 14.3 and 13.4; 3 of 64 7.1 and 7.0, 8.5 and 7.8, 9.5 and 8.7.
template <int DK, int DV, int HPB, bool BIAS, int KS>
__global__ void __launch_bounds__(HPB * 128 * KS, KS == 1 ? 2 : 1)
attn_prefill_kernel(AttnArgs a, const int4* __restrict__ tiles, int n_tiles) {
  constexpr int NT = HPB * 128 * KS, WAVES = NT / 64, SUBS = 2 / KS;
  constexpr int NSL = DK / 16, NDT = DV / 32;
  constexpr int KC = 64 * DK / 8 / NT, VC = 64 * DV / 8 / NT;
  constexpr float LOWEST = -3.4028234663852886e38f;
  __shared__ __attribute__((aligned(16))) short k0[64 * DK], k1[64 * DK];
  __shared__ __attribute__((aligned(16))) short v0[64 * DV], v1[64 * DV];
  __shared__ float other[KS > 1 ? HPB * 2 : 1][KS > 1 ? 16 * NDT + 2 : 1][64];

  const int tid = threadIdx.x, l = tid & 63;
  const int place = __builtin_amdgcn_readfirstlane(tid >> 6);      // among the waves
  const int wid = KS > 1 ? place >> 1 : place;                     // of a head's rows
  const int part = KS > 1 ? place & 1 : 0, k32 = 32 * part;        // of a page's keys
  const int lq = l & 31, half = l >> 5;
  int bx, by;
  xcd_tile_map(n_tiles, &bx, &by);
  bx = n_tiles - 1 - bx;               // a prompt's last tiles see most: first
  const int hg = a.H / a.G, nhc = hg / HPB;
  const int g = by / nhc;
  const int h = g * hg + (by % nhc) * HPB + (wid >> 1);
  const int4 t = tiles[bx];                    // first row, rows, pos0, slot
  const int row = 32 * (wid & 1) + lq;
  const int rowc = min(row, t.y - 1);
  const int ip = t.z + rowc, cs = first_seen(a, ip);

  bf16x8 qf[NSL];
  {
    const short* q = (const short*)a.qkv + (long)(t.x + rowc) * a.ld + (long)h * a.dim;
    #pragma unroll
    for (int s = 0; s < NSL; ++s) {
      const int c = 16 * s + 8 * half;
      qf[s] = c < a.dim ? *(const bf16x8*)(q + c) : bf16x8{};
    }
  }
  const int p_last = t.z + t.y - 1;
  const int first = first_seen(a, t.z) / LM_PAGE;
  const int n = p_last / LM_PAGE - first + 1;
  const int* tab = a.table + (long)t.w * a.max_pages + first;

  // this wave's rows: first and last position, and the last one's first key
  const int w0 = t.z + min(32 * (wid & 1), t.y - 1);
  const int w1 = t.z + min(32 * (wid & 1) + 31, t.y - 1);
  const bool w_any = 32 * (wid & 1) < t.y;
  const int wcs1 = first_seen(a, w1);

  // A lane's places in a page.  K image: rows with their 16-byte chunks XORed;
  // V image: units of 4 keys x 16 columns, for the transpose reads.
  constexpr unsigned NONE = 0x7ffffff0u;
  unsigned ko[KC], vo[VC];
  #pragma unroll
  for (int i = 0; i < KC; ++i) {
    const int s = i * NT + tid, j = s / (DK / 8);
    const int c = ((s % (DK / 8)) ^ (swapped(j) & 7)) * 8;
    ko[i] = c < a.dim ? 2u * (unsigned)(j * a.dim + c) : NONE;
  }
  #pragma unroll
  for (int i = 0; i < VC; ++i) {
    const int s = i * NT + tid, unit = s >> 3;
    const int j = 4 * (unit / (DV / 16)) + ((s >> 1) & 3);
    const int c = 16 * (unit % (DV / 16)) + 8 * (s & 1);
    vo[i] = c < a.vdim ? 2u * (unsigned)(j * a.vdim + c) : NONE;
  }
  auto copy = [&](auto count, short* to, const void* cache, int dim, const unsigned* at,
                  int page, int pg) INLINE {
    const unsigned long from =
        (unsigned long)((const short*)cache + ((long)page * a.G + g) * LM_PAGE * dim);
    const int rows = min(LM_PAGE, p_last - (first + pg) * LM_PAGE + 1);
    const auto src = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((unsigned long)same((unsigned)(from >> 32)) << 32 | same((unsigned)from)), 0,
        (int)same((unsigned)(2 * rows * dim)), 0x00020000);
    #pragma unroll
    for (int i = 0; i < decltype(count)::value; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          src, (__attribute__((address_space(3))) void*)(to + (i * WAVES + place) * 512),
          16, at[i], 0, 0, 0);
  };
  auto copy_k = [&](short* to, int page, int pg) INLINE {
    copy(std::integral_constant<int, KC>{}, to, a.kc, a.dim, ko, page, pg);
  };
  auto copy_v = [&](short* to, int page, int pg) INLINE {
    copy(std::integral_constant<int, VC>{}, to, a.vc, a.vdim, vo, page, pg);
  };
  // this wave's copies have arrived, in a form that the compiler's own count
  // takes notice of, and all waves are done with the page
  auto turn = []() INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  const float scale2 = a.scale * LOG2E;
  const float slope2 = BIAS && a.slopes ? a.slopes[h] * LOG2E : 0.f;
  const bool sink = a.has_sink && !part;
  float m_run = sink ? sink_score<false>(a, h) * LOG2E : LOWEST;
  if (m_run < LOWEST) m_run = LOWEST;          // -inf; NaN stays, and shows
  float l_run = sink && !half ? 1.f : 0.f;          // of this half's keys
  f32x16 o[NDT], s[SUBS];
  #pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = {};
  bf16x8 hi[SUBS][2], lo[SUBS][2];                  // weights, [sub][16 keys]

  auto scores = [&](const short* kimg) INLINE {
    #pragma unroll
    for (int sub = 0; sub < SUBS; ++sub) s[sub] = {};
    #pragma unroll
    for (int i = 0; i < NSL; ++i)
      #pragma unroll
      for (int sub = 0; sub < SUBS; ++sub)
        s[sub] = mma32(*(const bf16x8*)(kimg + (k32 + 32 * sub + swapped(lq)) * DK +
                                        ((2 * i + half) ^ (lq & 7)) * 8),
                       qf[i], s[sub]);
  };
  const int tr = 64 * (lq >> 4) + ((l & 15) >> 2) * 16 + (l & 3) * 4 +
                 (half ? 128 * (DV / 16) : 0) + k32 * DV;
  auto values = [&](const short* vimg) INLINE {
    typedef __attribute__((address_space(3))) bf16x4* P;
    auto quad = [&](int at) INLINE {
      return __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)(vimg + tr + at));
    };
    #pragma unroll
    for (int sub = 0; sub < SUBS; ++sub)
      #pragma unroll
      for (int i = 0; i < NDT; ++i)
        #pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int at = sub * 32 * DV + 64 * (4 * x * (DV / 16) + 2 * i);
          const bf16x8 vf = __builtin_shufflevector(
              quad(at), quad(at + 64 * (DV / 16)), 0, 1, 2, 3, 4, 5, 6, 7);
          o[i] = mma32(vf, hi[sub][x], o[i]);
          o[i] = mma32(vf, lo[sub][x], o[i]);
        }
  };
  auto softmax = [&](int j0) INLINE {
    const float d0 = slope2 * (float)(j0 + k32 + 8 * half - ip);
    #pragma unroll
    for (int sub = 0; sub < SUBS; ++sub)
      #pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int jr = 32 * sub + 16 * (r >> 3) + (r & 7);
        s[sub][r] *= scale2;
        if constexpr (BIAS) s[sub][r] += fmaf(slope2, (float)jr, d0);
      }
    if (j0 + LM_PAGE - 1 > w0 || j0 < wcs1) {
      asm volatile("");        // a branch, not 32 selects in every page
      const int from = cs - j0 - k32 - 8 * half, to = ip - j0 - k32 - 8 * half;
      #pragma unroll
      for (int sub = 0; sub < SUBS; ++sub)
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int jr = 32 * sub + 16 * (r >> 3) + (r & 7);
          if (jr < from || jr > to) s[sub][r] = -INFINITY;
        }
    }
    float top = s[0][0];
    #pragma unroll
    for (int sub = 0; sub < SUBS; ++sub)
      #pragma unroll
      for (int r = 0; r < 16; ++r) top = fmaxf(top, s[sub][r]);
    if (__any(top > m_run)) {
      top = over_halves(top, [](float x, float y) { return fmaxf(x, y); });
      const float mn = fmaxf(m_run, top);
      const float al = __builtin_amdgcn_exp2f(m_run - mn);
      m_run = mn;
      l_run *= al;
      #pragma unroll
      for (int i = 0; i < NDT; ++i)
        #pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= al;
    }
    float ps = 0.f;
    #pragma unroll
    for (int sub = 0; sub < SUBS; ++sub)
      #pragma unroll
      for (int x = 0; x < 2; ++x) {
        float e[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          e[j] = __builtin_amdgcn_exp2f(s[sub][8 * x + j] - m_run);
          ps += e[j];
        }
        union { unsigned u[4]; bf16x8 v; } p, q;
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          p.u[j] = cvt_pk_bf16(e[2 * j], e[2 * j + 1]);
          q.u[j] = cvt_pk_bf16(e[2 * j] - __builtin_bit_cast(float, p.u[j] << 16),
                               e[2 * j + 1] - __builtin_bit_cast(float, p.u[j] & 0xffff0000u));
        }
        hi[sub][x] = p.v;
        lo[sub][x] = q.v;
      }
    l_run += ps;
  };
  int now = tab[0], next = tab[min(1, n - 1)];     // pages' places
  auto page = [&](auto odd, auto begin, int it) INLINE {
    constexpr bool O = decltype(odd)::value;
    if (it + 1 < n) copy_k(O ? k0 : k1, next, it + 1);
    copy_v(O ? v1 : v0, now, it);
    now = next;
    next = tab[min(it + 2, n - 1)];
    if (w_any) {
      __builtin_amdgcn_s_setprio(1);
      scores(O ? k1 : k0);
      if constexpr (!decltype(begin)::value) values(O ? v0 : v1);
      // operands come from LDS four ahead of the product that takes them
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
      #pragma unroll
      for (int i = 0; i < SUBS * NSL - 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      if constexpr (!decltype(begin)::value) {
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        #pragma unroll
        for (int i = 0; i < 2 * SUBS * NDT - 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      softmax((first + it) * LM_PAGE);
    }
    turn();
  };
  constexpr std::true_type yes;
  constexpr std::false_type no;
  copy_k(k0, now, 0);
  turn();
  page(no, yes, 0);
  for (int it = 1; it < n; it += 2) {
    page(yes, no, it);
    if (it + 1 < n) page(no, no, it + 1);
  }
  if (KS == 1 && !w_any) return;
  if (n & 1) values(v0);
  else values(v1);

  l_run = over_halves(l_run, [](float x, float y) { return x + y; });
  if constexpr (KS > 1) {
    float(&to)[16 * NDT + 2][64] = other[wid];
    if (part) {
      #pragma unroll
      for (int i = 0; i < NDT; ++i)
        #pragma unroll
        for (int r = 0; r < 16; ++r) to[16 * i + r][l] = o[i][r];
      to[16 * NDT][l] = m_run;
      to[16 * NDT + 1][l] = l_run;
    }
    __syncthreads();
    if (part || !w_any) return;
    const float m1 = to[16 * NDT][l], mn = fmaxf(m_run, m1);
    // an infinite sink is the largest of all, and leaves nothing of what has scores
    const float al = __builtin_amdgcn_exp2f(m_run == mn ? 0.f : m_run - mn);
    const float be = __builtin_amdgcn_exp2f(m1 - mn);
    l_run = fmaf(l_run, al, to[16 * NDT + 1][l] * be);
    #pragma unroll
    for (int i = 0; i < NDT; ++i)
      #pragma unroll
      for (int r = 0; r < 16; ++r) o[i][r] = fmaf(o[i][r], al, to[16 * i + r][l] * be);
  }
  if (row < t.y) {
    const float inv = l_run > 0.f ? a.out_scale / l_run : 0.f;
    store_row<NDT>(a, o, inv, t.x + row, h, half);
  }
}

constexpr unsigned UNITS = 256;          // compute units

// pages that a tile sees at most
int most_pages(const AttnArgs& a) {
  const long reach = a.reach ? a.reach : (long)a.max_pages * LM_PAGE;
  const long seen = a.size ? std::min(reach, a.size + LM_PAGE - 1l) : reach;
  return (int)((seen + LM_PAGE - 1) / LM_PAGE);
}

// FORM 0: as stored; 1: with a bias by distance; 2: tied, with one; 3: window
template <int DK, int DV, int HPB, int FORM>
void go(const AttnArgs& a, const int4* tiles, int n, hipStream_t st) {
  const dim3 grid((unsigned)((long)n * a.G * (a.H / a.G / HPB)));
  if constexpr (FORM < 2) {
    if (grid.x <= UNITS && most_pages(a) >= (HPB == 2 ? 5 : DV / 64))
      hipLaunchKernelGGL((attn_prefill_kernel<DK, DV, HPB, FORM == 1, 2>), grid,
                         dim3(HPB * 256), 0, st, a, tiles, n);
    else
      hipLaunchKernelGGL((attn_prefill_kernel<DK, DV, HPB, FORM == 1, 1>), grid,
                         dim3(HPB * 128), 0, st, a, tiles, n);
  } else
    hipLaunchKernelGGL((attn_prefill_form_kernel<DK, DV, HPB, FORM == 2>), grid,
                       dim3(HPB * 128), 0, st, a, tiles, n);
}

template <int DK, int DV, int FORM>
void launch(const AttnArgs& a, const int4* tiles, int n, hipStream_t st) {
  const int hg = a.H / a.G;
  // Two blocks of 4 waves to a compute unit, which do not wait at each other's
  // barriers.  The window form spills with 4 waves.
  if constexpr (FORM >= 2) {
    if (hg % 4 == 0) return go<DK, DV, 4, FORM>(a, tiles, n, st);
  }
  if (hg % 2 == 0) go<DK, DV, 2, FORM>(a, tiles, n, st);
  else go<DK, DV, 1, FORM>(a, tiles, n, st);
}

template <int DK, int DV>
void pick_form(const AttnArgs& a, const int4* tiles, int n, hipStream_t st) {
  if (a.bias) launch<DK, DV, 3>(a, tiles, n, st);
  else if (a.slopes) launch<DK, DV, 1>(a, tiles, n, st);
  else launch<DK, DV, 0>(a, tiles, n, st);
}

}  // namespace

bool lm_attn_mfma_ok(const AttnArgs& a) {
  // rows of out that vectors can be stored to
  return a.dim % 8 == 0 && a.vdim % 8 == 0 && a.dim <= 128 && a.vdim <= 128 &&
         a.ldo % 4 == 0 && (size_t)a.out % 8 == 0;
}

void lm_attn_prefill_mfma(const AttnArgs& a, const int4* tiles, int n_tiles,
                          hipStream_t st) {
  if (a.ks) {
    if (a.dim <= 64) launch<64, 64, 2>(a, tiles, n_tiles, st);
    else launch<128, 128, 2>(a, tiles, n_tiles, st);
  } else if (a.dim <= 64) {
    if (a.vdim <= 64) pick_form<64, 64>(a, tiles, n_tiles, st);
    else pick_form<64, 128>(a, tiles, n_tiles, st);
  } else {
    if (a.vdim <= 64) pick_form<128, 64>(a, tiles, n_tiles, st);
    else pick_form<128, 128>(a, tiles, n_tiles, st);
  }
}
