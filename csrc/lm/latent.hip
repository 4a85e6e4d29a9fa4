// Latent attention (DeepSeek-AI, "DeepSeek-V2: A Strong, Economical, and
// Efficient Mixture-of-Experts Language Model"): a token caches one normed
// latent and one rotated key part that all heads share; a head's keys and
// values are products of the latent.
//
//   prep     norms of the query and key latents, rotation of the key part,
//            the append to the cache; gathers what the prompts see
//   prefill  attention over keys and values expanded from the gathered
//            latents (two GEMMs of the caller), queries rotated on load
//   decode   the key matrix moved to the query: 16 heads of a token against
//            the cached rows themselves, which serve as keys (all columns)
//            and values (the latent's columns); keys split over blocks,
//            up to 32 heads share them.
//            The value matrix and the head gates follow the merge.
//
// Scores, softmax and its weights are float; where the weights and the
// merged latents enter a bf16 product they go in as two parts.

#include "lm.h"
#include "tile.h"

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG = -1e30f;
constexpr int BLOCK = 128;      // prompt rows per block
constexpr int TABS = 1024;      // pages of a decode split

DEVINL int pad8(int n) { return (n + 7) & ~7; }

// rotate elements c..c+7 of a key part (pairs 2i, 2i+1) at position p
DEVINL void rotate8(float* v, int c, const LatentArgs& a, int p) {
  const int half = a.rd >> 1;
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = (c >> 1) + j;
    if (i < half) {
      const float cv = a.cos_t[(long)p * half + i], sv = a.sin_t[(long)p * half + i];
      const float x = v[2 * j], y = v[2 * j + 1];
      v[2 * j] = x * cv - y * sv;
      v[2 * j + 1] = y * cv + x * sv;
    }
  }
}

// dst = x * inv_rms(x) * w over n elements, one wave
template <bool F32, typename Put>
DEVINL void rms_row(const typename Num<F32>::E* x, const void* w, int n,
                    bool aligned, float eps, Put put) {
  const int l = threadIdx.x & 63;
  float q = 0.f;
  for (int c = l * 8; c < n; c += 512) {
    float v[8];
    load8<F32>(x + c, n - c, aligned, v);
    #pragma unroll
    for (int i = 0; i < 8; ++i) q += v[i] * v[i];
  }
  const float inv = 1.0f / sqrtf(group_sum<64>(q) / (float)n + eps);
  for (int c = l * 8; c < n; c += 512) {
    float v[8], g[8];
    load8<F32>(x + c, n - c, aligned, v);
    load8<F32>((const typename Num<F32>::E*)w + c, n - c, aligned, g);
    #pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= inv * g[i];
    put(c, v);
  }
}

// one wave per batch row, then one per gathered key
template <bool F32>
__global__ void __launch_bounds__(256)
latent_prep_kernel(LatentArgs a, const int* __restrict__ pos,
                   const int* __restrict__ slot, int T,
                   const void* __restrict__ qw, const void* __restrict__ kw,
                   void* __restrict__ cq, const int4* __restrict__ keys, int R,
                   void* __restrict__ c, void* __restrict__ kr) {
  using N = Num<F32>;
  using E = typename N::E;
  const long unit = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= (long)T + R) return;
  const int l = threadIdx.x & 63;
  const int roff = pad8(a.rank);
  const bool al = a.lda % 8 == 0 && a.q_rank % 8 == 0 && a.rank % 8 == 0;
  if (unit < T) {
    const int row = (int)unit, s = slot[row], p = pos[row];
    const E* src = (const E*)a.a + (long)row * a.lda;
    rms_row<F32>(src, qw, a.q_rank, al, a.eps, [&](int i, float* v) {
      store8<F32>((E*)cq + (long)row * a.q_rank + i, a.q_rank - i, al, v);
    });
    if (s < 0) return;
    const long page = a.table[(long)s * a.max_pages + p / LM_PAGE];
    E* cell = (E*)a.kc + (page * LM_PAGE + p % LM_PAGE) * a.row;
    // whole groups of 8: what pads the row is zero
    rms_row<F32>(src + a.q_rank, kw, a.rank, al, a.eps, [&](int i, float* v) {
      store8<F32>(cell + i, 8, true, v);
    });
    const int ri = l * 8;
    if (ri < a.row - roff) {
      float v[8];
      load8<F32>(src + a.q_rank + a.rank + ri, a.rot - ri, al && a.rot % 8 == 0, v);
      rotate8(v, ri, a, p);
      store8<F32>(cell + roff + ri, 8, true, v);
    }
    return;
  }
  const long key = unit - T;
  const int4 k = keys[key];                 // batch row or -1, slot, position
  E* cd = (E*)c + key * a.rank;
  E* kd = (E*)kr + key * a.rot;
  const bool ral = a.rot % 8 == 0;
  const int ri = l * 8;
  if (k.x >= 0) {
    const E* src = (const E*)a.a + (long)k.x * a.lda + a.q_rank;
    rms_row<F32>(src, kw, a.rank, al, a.eps, [&](int i, float* v) {
      store8<F32>(cd + i, a.rank - i, al, v);
    });
    if (ri < a.rot) {
      float v[8];
      load8<F32>(src + a.rank + ri, a.rot - ri, al && ral, v);
      rotate8(v, ri, a, k.z);
      store8<F32>(kd + ri, a.rot - ri, ral, v);
    }
  } else {
    const long page = a.table[(long)k.y * a.max_pages + k.z / LM_PAGE];
    const E* cell = (const E*)a.kc + (page * LM_PAGE + k.z % LM_PAGE) * a.row;
    for (int i = ri; i < a.rank; i += 512) {
      float v[8];
      load8<F32>(cell + i, 8, true, v);
      store8<F32>(cd + i, a.rank - i, a.rank % 8 == 0, v);
    }
    if (ri < a.rot) {
      float v[8];
      load8<F32>(cell + roff + ri, 8, true, v);
      store8<F32>(kd + ri, a.rot - ri, ral, v);
    }
  }
}

// Keep a load where it stands: the compiler would move it into a divergent
// branch of its one use, and every branch waits for its own load.
template <typename T> DEVINL void pin(T& v) { asm volatile("" : "+v"(v)); }

// Elements c..c+7 of a head's unrotated query part (ROT: rotated part, at
// position p); zeros past its end.  Aligned sizes take a path without
// divergent branches, so that all of a query's loads are in flight together.
template <bool F32, bool ROT>
DEVINL void load_query(const typename Num<F32>::E* q, int c, bool aligned,
                       const LatentArgs& a, int p, float* v) {
  const int n = ROT ? a.rot : a.dim;
  const typename Num<F32>::E* src = ROT ? q + a.dim : q;
  if (!aligned) {
    load8<F32>(src + c, n - c, false, v);
    if (ROT && c < a.rd) rotate8(v, c, a, p);
    return;
  }
  const bool in = c < n;
  float x[8];
  if constexpr (F32) {
    const f32x4 lo = *(const f32x4*)(q + (in ? (ROT ? a.dim : 0) + c : 0));
    const f32x4 hi = *(const f32x4*)(q + (in ? (ROT ? a.dim : 0) + c : 0) + 4);
    #pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = i < 4 ? lo[i & 3] : hi[i & 3];
  } else {
    const bf16x8 r = *(const bf16x8*)(q + (in ? (ROT ? a.dim : 0) + c : 0));
    #pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = bf2f(r[i]);
  }
  const int half = a.rd >> 1;
  if (ROT && half) {                        // uniform
    const float* ct = a.cos_t + (long)p * half;
    const float* st = a.sin_t + (long)p * half;
    float cs[4], sn[4];
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      cs[j] = ct[min((c >> 1) + j, half - 1)];
      sn[j] = st[min((c >> 1) + j, half - 1)];
    }
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      pin(cs[j]);
      pin(sn[j]);
    }
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool on = (c >> 1) + j < half;
      const float cv = on ? cs[j] : 1.f, sv = on ? sn[j] : 0.f;
      const float y = x[2 * j], z = x[2 * j + 1];
      x[2 * j] = y * cv - z * sv;
      x[2 * j + 1] = z * cv + y * sv;
    }
  }
  #pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = in ? x[i] : 0.f;
}

// the same 8 of a key, as stored: k its unrotated part, kr the rotated one
template <bool F32>
DEVINL void load_key(Raw8<F32>& r, const typename Num<F32>::E* k,
                     const typename Num<F32>::E* kr, int c, bool rot,
                     bool aligned, const LatentArgs& a) {
  if (rot) r.load(kr + c, a.rot - c, aligned);
  else r.load(k + c, a.dim - c, aligned);
}

DEVINL float head_gate(float z) { return 1.0f / (1.0f + expf(-z)); }

// ------------------------------------------------------- prompts, bf16
DEVINL unsigned pack2(float a, float b) {
  return (unsigned)(unsigned short)cvt_bf16(a) |
         ((unsigned)(unsigned short)cvt_bf16(b) << 16);
}

DEVINL f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, a),
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, b), c, 0,
      0, 0);
}

// B fragments (16 keys each) of 16 consecutive-by-lane P^T values
DEVINL void p_frags(const float* p, bf16x8 (&out)[2]) {
  #pragma unroll
  for (int s = 0; s < 2; ++s) {
    const unsigned ax = pack2(p[8 * s + 0], p[8 * s + 1]);
    const unsigned ay = pack2(p[8 * s + 2], p[8 * s + 3]);
    const unsigned bx = pack2(p[8 * s + 4], p[8 * s + 5]);
    const unsigned by = pack2(p[8 * s + 6], p[8 * s + 7]);
    auto rx = __builtin_amdgcn_permlane32_swap(ax, bx, false, false);
    auto ry = __builtin_amdgcn_permlane32_swap(ay, by, false, false);
    union { unsigned u[4]; bf16x8 v; } f;
    f.u[0] = rx[0]; f.u[1] = ry[0]; f.u[2] = rx[1]; f.u[3] = ry[1];
    out[s] = f.v;
  }
}

// A block is up to 128 prompt rows of one head, a wave 32 of them.  The
// layout of scores, weights and values is that of attn_mfma.hip: S^T = K Q^T,
// so that softmax is lane-local, and O^T = V^T P^T through the LDS transpose
// reads; keys come 64 at a time into a double buffer.
//
// A key's image is DU columns of its unrotated and DR of its rotated part.
// DIRECT (head sizes that are multiples of 8): keys and values go from
// memory to LDS without passing registers, each lane fetching what belongs
// in its 16 bytes of the images.  Columns that only pad an image get some
// other finite elements of the same token: the queries are zero there, and
// the values' are not stored.  The copies are issued after the score
// products, because LDS reads that the compiler sees wait for them.
template <int DU, int DR, int DV, bool DIRECT>
__global__ void __launch_bounds__(256, DU + DR + DV <= 320 ? 2 : 1)
latent_prefill_mfma_kernel(LatentArgs a, const short* __restrict__ q,
                           const short* __restrict__ k,
                           const short* __restrict__ v,
                           const short* __restrict__ kr,
                           const int4* __restrict__ blocks, int n_blocks,
                           short* __restrict__ out) {
  constexpr int NSL = (DU + DR) / 16, NDT = DV / 32;
  constexpr int BUF = 64 * (DU + DR + DV);     // two K images, V tr-image
  constexpr int UC = DU / 32, RC = DR / 32, VC = DV / 32;   // loads per thread
  extern __shared__ __attribute__((aligned(16))) short lds[];

  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  const int lq = l & 31, half = l >> 5;
  int bx, h;
  xcd_tile_map(n_blocks, &bx, &h);
  const int4 t = blocks[n_blocks - 1 - bx];    // the longest come first
  const int row = 32 * w + lq;
  const int rowc = min(row, t.y - 1);
  const int ip = t.z + rowc;
  const int size = a.size;
  constexpr bool aligned = DIRECT;             // what the launcher checked
  const long ldk = (long)a.H * a.dim, ldv = (long)a.H * a.vdim;

  bf16x8 qf[NSL];
  {
    const short* qr = q + ((long)(t.x + rowc) * a.H + h) * (a.dim + a.rot);
    #pragma unroll
    for (int s = 0; s < NSL; ++s) {
      float x[8];
      if (16 * s < DU) load_query<false, false>(qr, 16 * s + 8 * half, aligned, a, ip, x);
      else load_query<false, true>(qr, 16 * s - DU + 8 * half, aligned, a, ip, x);
      #pragma unroll
      for (int i = 0; i < 8; ++i) qf[s][i] = cvt_bf16(x[i]);
    }
  }

  const int p_last = t.z + t.y - 1;
  const int j_first = size ? max(0, t.z - size + 1) : 0;
  const int n_kt = (p_last - j_first) / 64 + 1;

  // this wave's rows: first and last position, first keys that they see
  const int w0 = t.z + min(32 * w, t.y - 1);
  const int w1 = t.z + min(32 * w + 31, t.y - 1);
  const bool w_any = 32 * w < t.y;
  const int lo0 = size ? w0 - size + 1 : 0, lo1 = size ? w1 - size + 1 : 0;
  const int lo = size ? ip - size + 1 : 0;

  const short* kh = k + (long)h * a.dim;
  const short* vh = v + (long)h * a.vdim;
  // DIRECT: a lane's column is the same in every pass over the tokens
  const int ju = tid / (DU / 8), jr = tid / (DR / 8);
  const int cu = ((tid % (DU / 8)) ^ (ju & 7)) * 8;
  const int cr = ((tid % (DR / 8)) ^ (jr & 7)) * 8;
  const int jv = 4 * (tid / (DV / 2)) + ((tid & 7) >> 1);
  const int cv = ((tid >> 3) % (DV / 16)) * 16 + (tid & 1) * 8;
  // (no rotated part at all: any readable address will do)
  const short* usrc = kh + (cu < a.dim ? cu : 0);
  const short* rsrc = a.rot ? kr + (cr < a.rot ? cr : 0) : kh;
  const short* vsrc = vh + (cv < a.vdim ? cv : 0);
  const long ldr = a.rot;
  auto stage_direct = [&](int j0, int buf) {
    short* ud = lds + buf * BUF + w * 512;
    short* rd = ud + 64 * DU;
    short* vd = rd + 64 * DR;
    #pragma unroll
    for (int i = 0; i < UC; ++i)
      glds16(usrc + ((long)t.w + min(j0 + i * (2048 / DU) + ju, p_last)) * ldk,
             ud + i * 2048);
    #pragma unroll
    for (int i = 0; i < RC; ++i)
      glds16(rsrc + ((long)t.w + min(j0 + i * (2048 / DR) + jr, p_last)) * ldr,
             rd + i * 2048);
    #pragma unroll
    for (int i = 0; i < VC; ++i)
      glds16(vsrc + ((long)t.w + min(j0 + i * (2048 / DV) + jv, p_last)) * ldv,
             vd + i * 2048);
  };
  Raw8<false> kreg[DIRECT ? 1 : UC + RC], vreg[DIRECT ? 1 : VC];
  auto stage_load = [&](int j0) {
    if constexpr (DIRECT) return;
    #pragma unroll
    for (int i = 0; i < UC + RC; ++i) {
      const bool rot = i >= UC;
      const int s = (rot ? i - UC : i) * 256 + tid, d8 = (rot ? DR : DU) / 8;
      const long key = (long)t.w + min(j0 + s / d8, p_last);
      load_key<false>(kreg[i], kh + key * ldk, kr + key * ldr, (s % d8) * 8,
                      rot, false, a);
    }
    #pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int s = i * 256 + tid, j = s / (DV / 8), c = (s % (DV / 8)) * 8;
      const long key = (long)t.w + min(j0 + j, p_last);
      vreg[i].load(vh + key * ldv + c, a.vdim - c, false);
    }
  };
  auto stage_write = [&](int buf) {
    if constexpr (DIRECT) return;
    short* kd = lds + buf * BUF;
    short* vd = kd + 64 * (DU + DR);
    #pragma unroll
    for (int i = 0; i < UC + RC; ++i) {
      const bool rot = i >= UC;
      const int s = (rot ? i - UC : i) * 256 + tid, d8 = (rot ? DR : DU) / 8;
      const int j = s / d8, cb = s % d8;
      *(bf16x8*)(kd + (rot ? 64 * DU : 0) + j * d8 * 8 + (cb ^ (j & 7)) * 8) =
          *(const bf16x8*)kreg[i].e;
    }
    #pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int s = i * 256 + tid, j = s / (DV / 8), c = (s % (DV / 8)) * 8;
      *(bf16x8*)(vd + ((j >> 2) * (DV / 16) + (c >> 4)) * 64 + (j & 3) * 16 +
                 (c & 15)) = *(const bf16x8*)vreg[i].e;
    }
  };
  const unsigned tr0 = lds_byte_off(lds + 64 * (DU + DR)) + 128u * (lq >> 4) +
                       ((l & 15) >> 2) * 32 + (l & 3) * 8 +
                       (half ? 128u * 2 * (DV / 16) : 0);

  const float scale2 = a.scale * LOG2E;
  float m_run = NEG, l_run = 0.f;
  f32x16 o[NDT];
  #pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = {};

  if constexpr (DIRECT) stage_direct(j_first, 0);
  stage_load(j_first);
  stage_write(0);
  __syncthreads();
  int cur = 0;
  for (int kt = 0; kt < n_kt; ++kt) {
    const int j0 = j_first + kt * 64;
    if (kt + 1 < n_kt) stage_load(j0 + 64);
    const bool seen = w_any && j0 <= w1 && j0 + 63 >= lo0;
    f32x16 s[2];
    s[0] = {};
    s[1] = {};
    if (seen) {
      const short* kimg = lds + cur * BUF;
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int kr_ = sub * 32 + lq;
        #pragma unroll
        for (int i = 0; i < DU / 16; ++i)
          s[sub] = mma32(*(const bf16x8*)(kimg + kr_ * DU +
                                          ((2 * i + half) ^ (kr_ & 7)) * 8),
                         qf[i], s[sub]);
        #pragma unroll
        for (int i = 0; i < DR / 16; ++i)
          s[sub] = mma32(*(const bf16x8*)(kimg + 64 * DU + kr_ * DR +
                                          ((2 * i + half) ^ (kr_ & 7)) * 8),
                         qf[DU / 16 + i], s[sub]);
      }
    }
    if constexpr (DIRECT) {
      if (kt + 1 < n_kt) stage_direct(j0 + 64, cur ^ 1);
    }
    if (seen) {
      const bool edge = j0 + 63 > w0 || j0 < lo1;
      float mt = NEG;
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          float x = s[sub][r] * scale2;
          if (edge) {
            const int j = j0 + sub * 32 + (r & 3) + 8 * (r >> 2) + 4 * half;
            x = fminf(x, (j <= ip) & (j >= lo) ? 3e38f : NEG);
          }
          s[sub][r] = x;
          mt = fmaxf(mt, x);
        }
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
      // The reference point moves only when scores pass it by 2^6: the
      // weights are floats, any common factor does.  A row that has seen
      // no key of its own yet collects finite junk here; its first own key
      // sets m_run and wipes it (alpha = 0).
      if (__any(mt > m_run + 6.f)) {
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
      l_run += ps + __shfl_xor(ps, 32, 64);

      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        float p[16], rem[16];
        #pragma unroll
        for (int r = 0; r < 16; ++r) p[r] = s[sub][r];
        bf16x8 hi[2], low[2];
        p_frags(p, hi);
        #pragma unroll
        for (int r = 0; r < 16; ++r) rem[r] = p[r] - bf2f(cvt_bf16(p[r]));
        p_frags(rem, low);
        const unsigned base = tr0 + (unsigned)cur * (BUF * 2) + (unsigned)sub * (32u * DV * 2);
        #pragma unroll
        for (int t2 = 0; t2 < NDT; t2 += 2) {
          auto addr = [&](int tt, int ss) {
            return base + 128u * (unsigned)((4 * ss) * (DV / 16) + 2 * tt);
          };
          const unsigned qs = 128u * (DV / 16);
          const bf16x8_quad x = tr_read_quad(
              addr(t2, 0), addr(t2, 0) + qs, addr(t2, 1), addr(t2, 1) + qs,
              addr(t2 + 1, 0), addr(t2 + 1, 0) + qs, addr(t2 + 1, 1),
              addr(t2 + 1, 1) + qs);
          o[t2] = mma32(x.f[0], hi[0], o[t2]);
          o[t2 + 1] = mma32(x.f[2], hi[0], o[t2 + 1]);
          o[t2] = mma32(x.f[1], hi[1], o[t2]);
          o[t2 + 1] = mma32(x.f[3], hi[1], o[t2 + 1]);
          o[t2] = mma32(x.f[0], low[0], o[t2]);
          o[t2 + 1] = mma32(x.f[2], low[0], o[t2 + 1]);
          o[t2] = mma32(x.f[1], low[1], o[t2]);
          o[t2 + 1] = mma32(x.f[3], low[1], o[t2 + 1]);
        }
      }
    }
    // the other buffer's readers passed the barrier of the last tile
    if (kt + 1 < n_kt) stage_write(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }

  if (row < t.y) {
    const float g = head_gate(bf2f(((const short*)a.a)[(long)(t.x + row) * a.lda +
                                                       a.q_rank + a.rank + a.rot + h]));
    const float inv = g / l_run;
    short* dst = out + (long)(t.x + row) * ldv + (long)h * a.vdim;
    #pragma unroll
    for (int i = 0; i < NDT; ++i)
      #pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int d = 32 * i + 8 * rq + 4 * half;
        if (aligned) {
          bf16x4 pk;
          #pragma unroll
          for (int j = 0; j < 4; ++j) pk[j] = cvt_bf16(o[i][rq * 4 + j] * inv);
          if (d < a.vdim) *(bf16x4*)(dst + d) = pk;
        } else {
          #pragma unroll
          for (int j = 0; j < 4; ++j)
            if (d + j < a.vdim) dst[d + j] = cvt_bf16(o[i][rq * 4 + j] * inv);
        }
      }
  }
}

// ---------------------------------------------------- prompts, float32
// 4 waves, 16 rows each: half a block of rows per workgroup
template <int DK, int DV>
__global__ void __launch_bounds__(256)
latent_prefill_f32_kernel(LatentArgs a, const float* __restrict__ q,
                          const float* __restrict__ k,
                          const float* __restrict__ v,
                          const float* __restrict__ kr,
                          const int4* __restrict__ blocks,
                          float* __restrict__ out) {
  using N = Num<true>;
  constexpr int LDK = DK + N::PAD, LDJ = 64 + N::PAD;
  extern __shared__ __attribute__((aligned(16))) float fl[];
  float* Ks = fl;                         // [64][LDK]
  float* Vt = Ks + 64 * LDK;              // [DV][LDJ]  values, transposed
  float* P = Vt + DV * LDJ;               // [64][LDJ]

  int4 t = blocks[blockIdx.x >> 1];
  const int off = (blockIdx.x & 1) * (BLOCK / 2);
  if (off >= t.y) return;
  t.x += off;
  t.z += off;
  t.y = min(t.y - off, BLOCK / 2);
  const int h = blockIdx.y;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int lr = l & 15, lg = l >> 4;
  const bool aligned = a.dim % 8 == 0 && a.vdim % 8 == 0 && a.rot % 8 == 0;
  const long ldk = (long)a.H * a.dim, ldv = (long)a.H * a.vdim;

  const int d8 = pad8(a.dim);             // where the rotated part starts
  N::Frag qf[DK / 32];
  {
    const int r = min(16 * w + lr, t.y - 1);
    const float* qr = q + ((long)(t.x + r) * a.H + h) * (a.dim + a.rot);
    #pragma unroll
    for (int kb = 0; kb < DK / 32; ++kb) {
      const int c = kb * 32 + lg * 8;
      if (c < d8) load_query<true, false>(qr, c, aligned, a, t.z + r, qf[kb].v);
      else load_query<true, true>(qr, c - d8, aligned, a, t.z + r, qf[kb].v);
    }
  }
  const float scale2 = a.scale * LOG2E;
  int lo[4], ip[4];
  float m[4], lsum[4];
  f32x4 o[DV / 16];
  #pragma unroll
  for (int i = 0; i < DV / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  #pragma unroll
  for (int r = 0; r < 4; ++r) {
    ip[r] = t.z + min(16 * w + 4 * lg + r, t.y - 1);
    lo[r] = a.size ? ip[r] - a.size + 1 : 0;
    m[r] = NEG;
    lsum[r] = 0.f;
  }
  const int p_last = t.z + t.y - 1;
  const int j_first = a.size ? max(0, t.z - a.size + 1) : 0;
  for (int j0 = j_first; j0 <= p_last; j0 += 64) {
    __syncthreads();                      // the last tile's reads are over
    for (int u = tid; u < 64 * (DK / 8); u += 256) {
      const int j = u / (DK / 8), c = (u % (DK / 8)) * 8;
      const long key = (long)t.w + min(j0 + j, p_last);
      Raw8<true> r;
      load_key<true>(r, k + key * ldk + (long)h * a.dim, kr + key * a.rot,
                     c < d8 ? c : c - d8, c >= d8, aligned, a);
      #pragma unroll
      for (int i = 0; i < 8; ++i) Ks[j * LDK + c + i] = r.e[i];
    }
    for (int u = tid; u < 64 * (DV / 8); u += 256) {
      const int j = u / (DV / 8), c = (u % (DV / 8)) * 8;
      const long key = (long)t.w + min(j0 + j, p_last);
      float x[8];
      load8<true>(v + key * ldv + (long)h * a.vdim + c, a.vdim - c, aligned, x);
      #pragma unroll
      for (int i = 0; i < 8; ++i) Vt[(c + i) * LDJ + j] = x[i];
    }
    __syncthreads();
    f32x4 s[4];
    #pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      s[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      #pragma unroll
      for (int kb = 0; kb < DK / 32; ++kb)
        s[ct] = N::mma(qf[kb], N::load(Ks + (ct * 16 + lr) * LDK, kb * 32 + lg * 8), s[ct]);
    }
    float al[4];
    #pragma unroll
    for (int r = 0; r < 4; ++r) {
      float mx = m[r];
      #pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        const int j = j0 + ct * 16 + lr;
        const bool ok = j <= ip[r] && j >= lo[r];
        s[ct][r] = ok ? s[ct][r] * scale2 : NEG;
        mx = fmaxf(mx, s[ct][r]);
      }
      mx = max16(mx);
      al[r] = exp2f(m[r] - mx);
      m[r] = mx;
      float e = 0.f;
      #pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        const float p = s[ct][r] > NEG ? exp2f(s[ct][r] - mx) : 0.f;
        P[(16 * w + 4 * lg + r) * LDJ + ct * 16 + lr] = p;
        e += p;
      }
      lsum[r] = lsum[r] * al[r] + sum16(e);
    }
    __syncthreads();
    #pragma unroll
    for (int i = 0; i < DV / 16; ++i)
      #pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] *= al[r];
    #pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const N::Frag pf = N::load(P + (16 * w + lr) * LDJ, kb * 32 + lg * 8);
      #pragma unroll
      for (int i = 0; i < DV / 16; ++i)
        o[i] = N::mma(pf, N::load(Vt + (i * 16 + lr) * LDJ, kb * 32 + lg * 8), o[i]);
    }
  }
  #pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * w + 4 * lg + r;
    if (row >= t.y) continue;
    const float g = head_gate(((const float*)a.a)[(long)(t.x + row) * a.lda + a.q_rank +
                                                  a.rank + a.rot + h]);
    const float inv = g / lsum[r];
    float* dst = out + (long)(t.x + row) * ldv + (long)h * a.vdim;
    #pragma unroll
    for (int i = 0; i < DV / 16; ++i)
      if (i * 16 + lr < a.vdim) dst[i * 16 + lr] = o[i][r] * inv;
  }
}

// ---------------------------------------------------------------- decode
// qa [R][H][row] = [W_uk^T q | rotated part]: 16 rows x 64 latent columns of
// one head per block
template <bool F32>
__global__ void __launch_bounds__(256)
latent_absorb_kernel(LatentArgs a, const void* __restrict__ q,
                     const void* __restrict__ wuk, const int* __restrict__ pos,
                     const int* __restrict__ slot, int R, float* __restrict__ qa) {
  using N = Num<F32>;
  using E = typename N::E;
  const int h = blockIdx.x, r0 = blockIdx.z * 16;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int lr = l & 15, lg = l >> 4;
  const int col = blockIdx.y * 64 + w * 16 + lr;
  const int hq = a.dim + a.rot;
  const bool al = a.dim % 8 == 0 && a.rot % 8 == 0;
  const E* qr = (const E*)q + ((long)min(r0 + lr, R - 1) * a.H + h) * hq;
  const E* wr = (const E*)wuk + (long)min(col, a.rank - 1) * a.H * a.dim + (long)h * a.dim;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < a.dim; kb += 32) {
    const int c = kb + lg * 8;
    Raw8<F32> x, y;
    x.load(qr + c, a.dim - c, al);
    y.load(wr + c, a.dim - c, al);
    acc = N::mma(N::load(x.e, 0), N::load(y.e, 0), acc);
  }
  if (col < a.rank) {
    #pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r0 + 4 * lg + r < R)
        qa[((long)(r0 + 4 * lg + r) * a.H + h) * a.row + col] = acc[r];
  }
  if (blockIdx.y) return;
  const int roff = pad8(a.rank), n8 = (a.row - roff) / 8;
  for (int u = tid; u < 16 * n8; u += 256) {
    const int row = r0 + u / n8, c = (u % n8) * 8;
    if (row >= R) continue;
    float v[8];
    load8<F32>((const E*)q + ((long)row * a.H + h) * hq + a.dim + c, a.rot - c, al, v);
    if (slot[row] >= 0) rotate8(v, c, a, pos[row]);
    float* d = qa + ((long)row * a.H + h) * a.row + roff + c;
    *(f32x4*)d = *(const f32x4*)v;
    *(f32x4*)(d + 4) = *(const f32x4*)(v + 4);
  }
  for (int u = tid; u < 16 * (roff - a.rank); u += 256) {
    const int row = r0 + u / (roff - a.rank);
    if (row < R) qa[((long)row * a.H + h) * a.row + a.rank + u % (roff - a.rank)] = 0.f;
  }
}

// A tile of cached rows in LDS, used as keys (row fragments) and as values
// (fragments along the tokens).  bf16: bands of 4 tokens in 4x16 subtiles,
// as the transpose reads want them; float: plain rows.
// RP: columns, a multiple of 32.
template <bool F32, int RP> struct RowTile {
  using N = Num<F32>;
  using E = typename N::E;
  static constexpr int KT = F32 ? 32 : 64;
  static constexpr int STRIDE = F32 ? RP + N::PAD : RP * 4 + 8;
  static constexpr int SIZE = F32 ? KT * STRIDE : KT / 4 * STRIDE;
  E* p;
  DEVINL E* at(int j, int c) const {        // c a multiple of 8
    if constexpr (F32) return p + j * STRIDE + c;
    else return p + (j >> 2) * STRIDE + (c >> 4) * 64 + (j & 3) * 16 + (c & 15);
  }
  DEVINL typename N::Frag row(int j, int c) const { return N::load(at(j, c), 0); }
  // column tiles ct..ct+CB-1 (16 each) of tokens 32*kb..+31
  template <int CB>
  DEVINL void cols(int ct, int kb, int l, typename N::Frag (&f)[CB]) const {
    static_assert(CB == 1 || CB == 2 || CB == 4, "columns at a time");
    const int lr = l & 15, lg = l >> 4;
    if constexpr (F32) {
      #pragma unroll
      for (int y = 0; y < CB; ++y)
        #pragma unroll
        for (int i = 0; i < 8; ++i)
          f[y].v[i] = p[(kb * 32 + lg * 8 + i) * STRIDE + (ct + y) * 16 + lr];
    } else {
      constexpr unsigned Q = 2u * STRIDE;
      const unsigned s = lds_byte_off(p) + (unsigned)(kb * 8 + 2 * lg) * Q +
                         (unsigned)ct * 128u + (lr >> 2) * 32 + (lr & 3) * 8;
      if constexpr (CB == 1) {
        f[0] = tr_read_frag(s, s + Q);
      } else if constexpr (CB == 2) {
        const bf16x8_pair r = tr_read_pair(s, s + Q, s + 128, s + Q + 128);
        f[0] = r.f[0];
        f[1] = r.f[1];
      } else {
        const bf16x8_quad r = tr_read_quad(s, s + Q, s + 128, s + Q + 128,
                                           s + 256, s + Q + 256, s + 384,
                                           s + Q + 384);
        #pragma unroll
        for (int y = 0; y < 4; ++y) f[y] = r.f[y];
      }
    }
  }
};

template <bool F32, int NC, int HG>
constexpr int decode_lds() {                // bytes of dynamic LDS
  using N = Num<F32>;
  using T = RowTile<F32, 64 * NC + 64>;
  return (int)sizeof(typename N::E) *
         (2 * T::SIZE + HG * Split<F32>::PARTS * 16 * (T::KT + N::PAD));
}

// grid: split, HG groups of 16 heads, row.  Four waves a group: each scores
// a quarter of the tile's tokens (float: half, two waves) with its queries
// in registers and sums a quarter of the latent's columns, NC of 16.  The
// groups share the tile; the next one waits in registers for the other
// buffer.
template <bool F32, int NC, int HG>
__global__ void __launch_bounds__(256 * HG)
latent_decode_kernel(LatentArgs a, const float* __restrict__ qa,
                     const int* __restrict__ pos, const int* __restrict__ slot,
                     int nsplit, float* __restrict__ ws) {
  using N = Num<F32>;
  using E = typename N::E;
  constexpr int ROW = 64 * NC + 64;         // the longest row of the class
  using Tile = RowTile<F32, ROW>;
  constexpr int KT = Tile::KT, NT = 256 * HG;
  constexpr int LPT = NT / KT;              // lanes that share a token's row
  constexpr int NL = (ROW / 8 + LPT - 1) / LPT;       // loads per thread
  constexpr int NKB = ROW / 32;
  constexpr int LDP = KT + N::PAD;
  constexpr int KW = KT / 16;               // waves of a group that score
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float m_s[2][HG][4][16], l_s[HG][4][16];
  __shared__ int tab_s[TABS];

  const int split = blockIdx.x, b = blockIdx.z;
  const int s = slot[b];
  if (s < 0) return;                        // the merge skips the row as well
  const int tid = threadIdx.x, l = tid & 63;
  const int w = (tid >> 6) & 3, g = tid >> 8;
  const int lr = l & 15, lg = l >> 4;
  E* tiles = (E*)smem;
  E* pb = tiles + 2 * Tile::SIZE + g * Split<F32>::PARTS * 16 * LDP;
  const Split<F32> P{pb, pb + 16 * LDP};
  const int h0 = (blockIdx.y * HG + g) * 16;
  const int nh = min(16, a.H - h0);         // may be <= 0 in the last block

  const int p = pos[b];
  const int first = a.size ? max(0, p - a.size + 1) : 0;
  const int per = ((p - first + nsplit) / nsplit + KT - 1) / KT * KT;
  const int jb = first + split * per, je = min(jb + per, p + 1);
  float* dst = ws + (((long)b * a.H + h0) * nsplit + split) * (a.rank + 2);
  const long hstep = (long)nsplit * (a.rank + 2);
  if (jb >= je) {                           // nothing left for this split
    for (int i = 0; i < nh; ++i)
      for (int c = tid & 255; c < a.rank + 2; c += 256)
        dst[i * hstep + c] = c ? 0.f : NEG;
    return;
  }
  const int* tab = a.table + (long)s * a.max_pages;
  const int pg0 = jb / LM_PAGE, npg = (je - 1) / LM_PAGE - pg0 + 1;
  for (int i = tid; i < npg; i += NT) tab_s[i] = tab[pg0 + i];
  // queries, zeros past the row and the heads
  typename N::Frag qf[NKB];
  #pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    const int c = kb * 32 + lg * 8;
    const bool on = lr < nh && c < a.row;
    Raw8<true> v;
    v.load(on ? qa + ((long)b * a.H + h0 + lr) * a.row + c : qa, 8, true);
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = on ? v[i] : 0.f;
      if constexpr (F32) qf[kb].v[i] = x;
      else qf[kb][i] = cvt_bf16(x);
    }
    if (kb % 6 == 5) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  // a thread moves every LPT-th 8 elements of one token; columns past the
  // row get its last ones again, the query is zero there
  const int jt = tid / LPT, c0 = tid % LPT * 8;
  Raw8<F32> r[NL];
  auto fetch = [&](int j0) {                // tokens past the end: the last
    const int j = min(j0 + jt, je - 1);
    const E* src = (const E*)a.kc +
                   ((long)tab_s[j / LM_PAGE - pg0] * LM_PAGE + j % LM_PAGE) * a.row;
    #pragma unroll
    for (int i = 0; i < NL; ++i)
      r[i].load(src + min(c0 + i * LPT * 8, a.row - 8), 8, true);
  };
  auto put = [&](int buf) {
    const Tile K{tiles + buf * Tile::SIZE};
    #pragma unroll
    for (int i = 0; i < NL; ++i) {
      if (c0 + i * LPT * 8 >= ROW) continue;  // LPT may not divide the row
      E* d = K.at(jt, c0 + i * LPT * 8);
      if constexpr (F32) {
        *(f32x4*)d = *(const f32x4*)r[i].e;
        *(f32x4*)(d + 4) = *(const f32x4*)(r[i].e + 4);
      } else {
        *(bf16x8*)d = *(const bf16x8*)r[i].e;
      }
    }
  };

  const float scale2 = a.scale * LOG2E;
  float m[4], ls[4];
  f32x4 o[NC];
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    m[i] = NEG;
    ls[i] = 0.f;
  }
  #pragma unroll
  for (int i = 0; i < NC; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(jb);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = jb; j0 < je; j0 += KT, buf ^= 1) {
    const Tile K{tiles + buf * Tile::SIZE};
    const bool more = j0 + KT < je;
    if (more) fetch(j0 + KT);
    f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool ok = w < KW && j0 + 16 * w + lr < je;
    if (w < KW) {
      #pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        sc = N::mma(qf[kb], K.row(16 * w + lr, kb * 32 + lg * 8), sc);
        // six fragments in flight, not all: the registers are needed
        if (kb % 6 == 5) __builtin_amdgcn_sched_barrier(0);
      }
    }
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[i] = ok ? sc[i] * scale2 : NEG;
      const float x = max16(sc[i]);
      if (lr == 0) m_s[buf][g][w][4 * lg + i] = x;
    }
    __syncthreads();
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mn = m[i];
      #pragma unroll
      for (int x = 0; x < KW; ++x) mn = fmaxf(mn, m_s[buf][g][x][4 * lg + i]);
      const float al = exp2f(m[i] - mn);
      const float e = ok ? exp2f(sc[i] - mn) : 0.f;
      m[i] = mn;
      ls[i] = ls[i] * al + e;
      if (w < KW) P.put((4 * lg + i) * LDP + 16 * w + lr, e);
      #pragma unroll
      for (int x = 0; x < NC; ++x) o[x][i] *= al;
    }
    __syncthreads();
    #pragma unroll
    for (int kb = 0; kb < KT / 32; ++kb) {
      const auto pf = P.load(lr * LDP, kb * 32 + lg * 8);
      constexpr int CB = NC % 4 == 0 ? 4 : NC;          // columns at a time
      #pragma unroll
      for (int x = 0; x < NC; x += CB) {
        typename N::Frag f[CB];
        K.template cols<CB>(w * NC + x, kb, l, f);
        #pragma unroll
        for (int y = 0; y < CB; ++y) o[x + y] = mma_sp<F32>(pf, f[y], o[x + y]);
      }
    }
    // the other buffer's readers passed this barrier a tile ago
    if (more) put(buf ^ 1);
    __syncthreads();
  }
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = sum16(ls[i]);
    if (lr == 0) l_s[g][w][4 * lg + i] = x;
  }
  __syncthreads();
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int hh = 4 * lg + i;
    if (hh >= nh) continue;
    float* d = dst + hh * hstep;
    if (w == 0 && lr == 0) {
      d[0] = m[i];
      d[1] = l_s[g][0][hh] + l_s[g][1][hh] + l_s[g][2][hh] + l_s[g][3][hh];
    }
    #pragma unroll
    for (int x = 0; x < NC; ++x) {
      const int c = (w * NC + x) * 16 + lr;
      if (c < a.rank) d[2 + c] = o[x][i];
    }
  }
}

// Merge of the splits, value matrix and gate: 16 rows x 128 value columns
// of one head per block
template <bool F32>
__global__ void __launch_bounds__(512)
latent_out_kernel(LatentArgs a, const float* __restrict__ ws,
                  const void* __restrict__ wuv, const int* __restrict__ slot,
                  int R, int nsplit, void* __restrict__ out) {
  using N = Num<F32>;
  using E = typename N::E;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float f_s[16][64];
  const int h = blockIdx.x, r0 = blockIdx.z * 16;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int lr = l & 15, lg = l >> 4;
  const int rp = (a.rank + 31) & ~31, ld = rp + N::PAD;
  const Split<F32> L{(E*)smem, (E*)smem + 16 * ld};
  const int st = a.rank + 2;
  if (tid < 256) {
    // 16 lanes weigh a row's splits (at most 64), four each
    const int i = tid >> 4, x0 = tid & 15, row = r0 + i;
    const bool on = row < R && slot[min(row, R - 1)] >= 0;
    const float* p = ws + ((long)min(row, R - 1) * a.H + h) * nsplit * st;
    float m[4], s[4], mx = NEG, lt = 0.f;
    #pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int x = x0 + 16 * y;
      m[y] = on && x < nsplit ? p[(long)x * st] : NEG;
      s[y] = on && x < nsplit ? p[(long)x * st + 1] : 0.f;
      mx = fmaxf(mx, m[y]);
    }
    mx = max16(mx);
    #pragma unroll
    for (int y = 0; y < 4; ++y) {
      m[y] = s[y] > 0.f ? exp2f(m[y] - mx) : 0.f;
      lt += m[y] * s[y];
    }
    lt = sum16(lt);
    #pragma unroll
    for (int y = 0; y < 4; ++y) f_s[i][x0 + 16 * y] = lt > 0.f ? m[y] / lt : 0.f;
  }
  __syncthreads();
  // 32 lanes a row, many loads in flight before they are used; an idle
  // row's partial results were never written
  {
    const int i = tid >> 5, row = r0 + i;
    const bool on = row < R && slot[min(row, R - 1)] >= 0;
    const float* p = ws + ((long)min(row, R - 1) * a.H + h) * nsplit * st + 2;
    constexpr int CU = 8;
    for (int c0 = tid & 31; c0 < rp; c0 += 32 * CU) {
      float x[CU];
      #pragma unroll
      for (int y = 0; y < CU; ++y) x[y] = 0.f;
      #pragma unroll 4
      for (int z = 0; z < (on ? nsplit : 0); ++z) {
        const float f = f_s[i][z];
        float v[CU];
        #pragma unroll
        for (int y = 0; y < CU; ++y)
          v[y] = p[(long)z * st + min(c0 + 32 * y, a.rank - 1)];
        #pragma unroll
        for (int y = 0; y < CU; ++y) x[y] = fmaf(f, v[y], x[y]);
      }
      #pragma unroll
      for (int y = 0; y < CU; ++y) {
        const int c = c0 + 32 * y;
        if (c < rp) L.put(i * ld + c, c < a.rank ? x[y] : 0.f);
      }
    }
  }
  __syncthreads();
  const int e = blockIdx.y * 128 + w * 16 + lr;
  const bool al = a.rank % 8 == 0;
  const E* wr = (const E*)wuv + ((long)h * a.vdim + min(e, a.vdim - 1)) * a.rank;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  #pragma unroll 8
  for (int kb = 0; kb < rp; kb += 32) {
    const int c = kb + lg * 8;
    Raw8<F32> y;
    y.load(wr + c, a.rank - c, al);
    acc = mma_sp<F32>(L.load(lr * ld, c), N::load(y.e, 0), acc);
  }
  if (e >= a.vdim) return;
  #pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = r0 + 4 * lg + r;
    if (row >= R) continue;
    const float g = head_gate(N::up(((const E*)a.a)[(long)row * a.lda + a.q_rank +
                                                    a.rank + a.rot + h]));
    ((E*)out)[((long)row * a.H + h) * a.vdim + e] = N::down(acc[r] * g);
  }
}

template <int DU, int DR, int DV, bool DIRECT>
void go_mfma(const LatentArgs& a, const void* q, const void* k, const void* v,
             const void* kr, const int4* blocks, int n, void* out,
             hipStream_t st) {
  constexpr int lds = 2 * 64 * (DU + DR + DV) * 2;
  static_assert(lds <= 160 * 1024, "exceeds the CU's LDS");
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)latent_prefill_mfma_kernel<DU, DR, DV, DIRECT>,
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  hipLaunchKernelGGL((latent_prefill_mfma_kernel<DU, DR, DV, DIRECT>),
                     dim3((unsigned)((long)n * a.H)), dim3(256), lds, st, a,
                     (const short*)q, (const short*)k, (const short*)v,
                     (const short*)kr, blocks, n, (short*)out);
}

template <int DU, int DR>
void mfma_dv(const LatentArgs& a, const void* q, const void* k, const void* v,
             const void* kr, const int4* blocks, int n, void* out,
             hipStream_t st) {
  if (a.vdim <= 64) go_mfma<DU, DR, 64, true>(a, q, k, v, kr, blocks, n, out, st);
  else if (a.vdim <= 128) go_mfma<DU, DR, 128, true>(a, q, k, v, kr, blocks, n, out, st);
  else go_mfma<DU, DR, 256, true>(a, q, k, v, kr, blocks, n, out, st);
}

void run_mfma(const LatentArgs& a, const void* q, const void* k, const void* v,
              const void* kr, const int4* blocks, int n, void* out,
              hipStream_t st) {
  if (a.dim > 128 && a.rot > 64)
    go_mfma<192, 128, 256, false>(a, q, k, v, kr, blocks, n, out, st);
  else if (a.dim % 8 || a.vdim % 8 || a.rot % 8) {
    if (a.dim <= 128 && a.vdim <= 128)
      go_mfma<128, 128, 128, false>(a, q, k, v, kr, blocks, n, out, st);
    else if (a.dim <= 128)
      go_mfma<128, 128, 256, false>(a, q, k, v, kr, blocks, n, out, st);
    else
      go_mfma<256, 64, 256, false>(a, q, k, v, kr, blocks, n, out, st);
  } else if (a.dim > 128) mfma_dv<256, 64>(a, q, k, v, kr, blocks, n, out, st);
  else if (a.rot > 64) mfma_dv<128, 128>(a, q, k, v, kr, blocks, n, out, st);
  else if (a.dim > 64) mfma_dv<128, 64>(a, q, k, v, kr, blocks, n, out, st);
  else mfma_dv<64, 64>(a, q, k, v, kr, blocks, n, out, st);
}

template <int DK, int DV>
void go_f32(const LatentArgs& a, const void* q, const void* k, const void* v,
            const void* kr, const int4* blocks, int n, void* out,
            hipStream_t st) {
  constexpr int lds = 4 * (64 * (DK + 4) + (DV + 64) * 68);
  static_assert(lds <= 160 * 1024, "exceeds the CU's LDS");
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)latent_prefill_f32_kernel<DK, DV>,
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  hipLaunchKernelGGL((latent_prefill_f32_kernel<DK, DV>), dim3(2 * n, a.H),
                     dim3(256), lds, st, a, (const float*)q, (const float*)k,
                     (const float*)v, (const float*)kr, blocks, (float*)out);
}

template <bool F32, int NC, int HG>
void go_decode_as(const LatentArgs& a, const int* pos, const int* slot, int R,
                  int nsplit, const float* qa, float* ws, hipStream_t st) {
  constexpr int lds = decode_lds<F32, NC, HG>();
  static_assert(lds <= 153 * 1024 + 512, "exceeds the CU's LDS");
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)latent_decode_kernel<F32, NC, HG>,
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  hipLaunchKernelGGL((latent_decode_kernel<F32, NC, HG>),
                     dim3(nsplit, (a.H + 16 * HG - 1) / (16 * HG), R),
                     dim3(256 * HG), lds, st, a, qa, pos, slot, nsplit, ws);
}

template <bool F32, int NC>
void go_decode(const LatentArgs& a, const int* pos, const int* slot, int R,
               int nsplit, const float* qa, float* ws, hipStream_t st) {
  if (a.H <= 16) go_decode_as<F32, NC, 1>(a, pos, slot, R, nsplit, qa, ws, st);
  else go_decode_as<F32, NC, 2>(a, pos, slot, R, nsplit, qa, ws, st);
}

template <bool F32>
void run_decode(const LatentArgs& a, const void* q, const void* wuk,
                const void* wuv, const int* pos, const int* slot, int R,
                int nsplit, float* qa, float* ws, void* out, hipStream_t st) {
  const int rg = (R + 15) / 16;
  hipLaunchKernelGGL((latent_absorb_kernel<F32>),
                     dim3(a.H, (a.rank + 63) / 64, rg), dim3(256), 0, st, a, q,
                     wuk, pos, slot, R, qa);
  // a class serves ranks up to 64 NC and rows up to 64 (NC + 1)
  const int nc = std::max((a.rank + 63) / 64, (a.row + 63) / 64 - 1);
  if (nc <= 1) go_decode<F32, 1>(a, pos, slot, R, nsplit, qa, ws, st);
  else if (nc <= 2) go_decode<F32, 2>(a, pos, slot, R, nsplit, qa, ws, st);
  else if (nc <= 4) go_decode<F32, 4>(a, pos, slot, R, nsplit, qa, ws, st);
  else go_decode<F32, 8>(a, pos, slot, R, nsplit, qa, ws, st);
  using N = Num<F32>;
  const int lds = (int)sizeof(typename N::E) * Split<F32>::PARTS * 16 *
                  (((a.rank + 31) & ~31) + N::PAD);
  hipLaunchKernelGGL((latent_out_kernel<F32>), dim3(a.H, (a.vdim + 127) / 128, rg),
                     dim3(512), lds, st, a, (const float*)ws, wuv, slot, R,
                     nsplit, out);
}

}  // namespace

void lm_latent_prep(const LatentArgs& a, const int* pos, const int* slot,
                    int T, const void* qw, const void* kw, void* cq,
                    const int4* keys, int R, void* c, void* kr, bool f32,
                    hipStream_t stream) {
  const long units = (long)T + R;
  if (units <= 0) return;
  const dim3 grid((unsigned)((units + 3) / 4));
  if (f32)
    hipLaunchKernelGGL((latent_prep_kernel<true>), grid, dim3(256), 0, stream,
                       a, pos, slot, T, qw, kw, cq, keys, R, c, kr);
  else
    hipLaunchKernelGGL((latent_prep_kernel<false>), grid, dim3(256), 0, stream,
                       a, pos, slot, T, qw, kw, cq, keys, R, c, kr);
}

void lm_latent_prefill(const LatentArgs& a, const void* q, const void* k,
                       const void* v, const void* kr, const int4* blocks,
                       int n_blocks, void* out, bool f32, hipStream_t stream) {
  if (n_blocks <= 0) return;
  if (!f32) {
    run_mfma(a, q, k, v, kr, blocks, n_blocks, out, stream);
    return;
  }
  const int dk = ((a.dim + 7) & ~7) + ((a.rot + 7) & ~7);
  #define LP_GO(DK, DV) go_f32<DK, DV>(a, q, k, v, kr, blocks, n_blocks, out, stream)
  if (dk <= 64 && a.vdim <= 64) LP_GO(64, 64);
  else if (dk <= 128 && a.vdim <= 128) LP_GO(128, 128);
  else LP_GO(256, 256);
  #undef LP_GO
}

bool lm_latent_decode_fits(const LatentArgs& a) {
  return a.rank <= 512 && a.row <= 576;
}

void lm_latent_decode(const LatentArgs& a, const void* q, const void* wuk,
                      const void* wuv, const int* pos, const int* slot, int R,
                      int nsplit, float* qa, float* ws, void* out, bool f32,
                      hipStream_t stream) {
  if (R <= 0) return;
  if (f32) run_decode<true>(a, q, wuk, wuv, pos, slot, R, nsplit, qa, ws, out, stream);
  else run_decode<false>(a, q, wuk, wuv, pos, slot, R, nsplit, qa, ws, out, stream);
}
