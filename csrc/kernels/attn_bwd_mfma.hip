// K4 — MFMA flash attention backward (bf16, CDNA4 32x32x16), from the forward's
// logsumexp.  A wave has 32 rows, whose operands and sums stay in registers; the
// others come through LDS in tiles of 64:
//
//  dQ      wave = 32 query rows, tiles of K and V
//    S^T  = K Q^T, dP^T = V dO^T             lane = query, registers = keys
//    dS^T = P^T (dP^T - delta) scale,  dQ^T += K^T dS^T
//  dK, dV  wave = 32 key rows, tiles of Q and dO, over the heads that share them
//    S = Q K^T, dP = dO V^T                  lane = key, registers = queries
//    dV += P^T dO,  dK += dS^T Q
//
//  * An image of a tile is read by rows (16 bytes a lane) and by columns
//    (transpose reads): its chunks of 8 columns are XORed so that neither has
//    bank conflicts.  In images of 4 x 16 units, which suit the transpose reads
//    alone, four of eight lanes of a row read met in a bank.
//  * Blocks of 4 waves, two or more to a compute unit, that nothing ties to
//    each other: while one multiplies, another has its exponentials.  Copies go
//    to images that are arrays of their own, so that the compiler knows that
//    a read of one need not wait for copies into another.  Blocks of all heads
//    start in order of length.
//  * dK and dV of heads of 128 take 192 registers for operands and sums alone:
//    with two waves to a SIMD no room is left to have operands on their way, and
//    the products wait for each read of LDS (996 us instead of 633).  There is one wave
//    then, with its products, reads and weights laid one between the other.
//
// What bounds it: dK and dV of heads of 128 vector work (1.3 cycles for each of
// the matrix cores', of which 64 of 350 instructions fetch scores from
// accumulators) and the first reads of a tile; the others waits, the matrix
// cores being busy 22 to 45 % of the time.
//
// In us, dQ + dK and dV, against blocks of 8 waves (heads of 64), waves of two
// roles for dK and dV and a dQ of unequal ends (128), 4 x 16 images:
//   16 x 12 x 1024 x 64            62 +  89   106 + 157
//   3 x 12 x 333 x 64              10 +  17    19 +  23
//   2 x 32 (8 kv) x 4096 x 128    388 + 633   723 + 955
//   1 x 32 (8 kv) x 512 x 128      19 +  72   132 in all
// The sums run over the same products in the same order, bit by bit.

#include "../common.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short bf16x8_t __attribute__((ext_vector_type(8)));

constexpr float LOG2E = 1.4426950408889634f;
constexpr int ROWS = 128;              // of a block of 4 waves

// What a lane holds of a product's 32 x 32 (a column, 16 rows), as operands of
// 8 consecutive rows a lane: the halves exchange every other four.
DEVINL bf16x8_t exchange(const unsigned* w) {
  const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  union { unsigned u[4]; bf16x8_t v; } f = {{x[0], y[0], x[1], y[1]}};
  return f.v;
}

DEVINL void pack_frags(const f32x16_t& p, bf16x8_t out[2]) {
  #pragma unroll
  for (int s = 0; s < 2; ++s) {
    unsigned w[4];
    #pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = cvt_pk_bf16(p[8 * s + 2 * j], p[8 * s + 2 * j + 1]);
    out[s] = exchange(w);
  }
}

DEVINL f32x16_t mma(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Image of 64 rows of D: element (row, col) is at row * D + 8 * ((col / 8) ^
// chunk_key(row)) + col % 8.  Eight (D 64) or sixteen consecutive rows have the
// same chunk in different places, four have the same pair of chunks in
// different pairs.
template <int D>
DEVINL int chunk_key(int row) {
  if constexpr (D == 64) return (row & 3) << 1 | ((row >> 2) & 1);
  else return (row & 7) << 1 | ((row >> 3) & 1);
}

template <int D>
struct Image {
  int row0, col0;

  DEVINL explicit Image(int l) {
    const int lq = l & 31, half = l >> 5, r = (l & 15) >> 2;
    row0 = lq * D + 8 * (half ^ chunk_key<D>(lq));
    col0 = (8 * half + r) * D + 4 * (l & 1) +
           8 * ((2 * (lq >> 4) + ((l & 3) >> 1)) ^ (r << 1) ^ (D == 128 ? half : 0));
  }
  // The same, but not known to be: what is computed from it is computed again
  // in each tile, a cycle or two, instead of kept in a register for each place.
  DEVINL Image again() const {
    Image i = *this;
    asm volatile("" : "+v"(i.row0), "+v"(i.col0));
    return i;
  }
  // columns 16 s + 8 half ... of row 32 sub + lq
  DEVINL bf16x8_t row(const short* img, int sub, int s) const {
    return *(const bf16x8_t*)(img + 32 * sub * D + (row0 ^ (16 * s)));
  }
  // rows 32 sub + 16 s + 8 half ... of column 32 t + lq
  DEVINL bf16x8_t col(const short* img, int sub, int t, int s) const {
    typedef __attribute__((address_space(3))) bf16x4* P;
    auto quad = [&](int q) INLINE {
      return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (P)(img + (32 * sub + 16 * s + 4 * q) * D +
              (col0 ^ (8 * ((4 * t) ^ (D == 64 ? q : 8 * q))))));
    };
    return __builtin_shufflevector(quad(0), quad(1), 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// Copies rows r0 ... r0 + 63 of a tensor into an image, by buffer loads: rows
// from S on read as zero.  lane_at: this lane's place in the first rows.
template <int D>
DEVINL unsigned copy_at(long ss) {
  const int row = threadIdx.x / (D / 8), chunk = threadIdx.x % (D / 8);
  return 2u * ((unsigned)row * (unsigned)ss + 8u * (chunk ^ chunk_key<D>(row)));
}

template <int D>
DEVINL void copy_rows(short* img, const short* from, long ss, unsigned lane_at,
                      int r0, int S, int wid) {
  constexpr int STEP = 256 / (D / 8);  // rows that the block copies at once
  static_assert(STEP % 16 == 0, "chunk_key() must be the same in every step");
  asm volatile("" : "+v"(lane_at));    // steps are added, not kept
  const long last = min(64, S - r0) - 1;
  const unsigned long at = (unsigned long)(from + (long)r0 * ss);
  const auto rows = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((unsigned long)same((unsigned)(at >> 32)) << 32 | same((unsigned)at)), 0,
      (int)same((unsigned)((last * ss + D) * 2)), 0x00020000);
  #pragma unroll
  for (int i = 0; i < 64 / STEP; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (__attribute__((address_space(3))) void*)(img + (i * 4 + wid) * 512),
        16, lane_at + i * STEP * 2u * (unsigned)ss, 0, 0, 0);
}

// the copies of this wave have arrived, in a form that the compiler's own
// count takes notice of, and every wave is done with the tile
DEVINL void next_tile() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// delta = rowsum(dO * O) - dlse, D/8 lanes a row (stride-aware): bound by
// reading both once, so every lane has 16 bytes of each.
// dlse (may be null) is the gradient of the attention's logsumexp
// output — context-parallel partial-attention merges differentiate
// through lse (scaffold/dist/cp.py); folding it here makes the dq/dkv
// kernels' (dP - delta) term exact with zero extra passes.
template <int D>
__global__ void __launch_bounds__(256)
attn_delta_strided_kernel(const short* __restrict__ dout,
                          const short* __restrict__ o,
                          const float* __restrict__ dlse,
                          float* __restrict__ delta, int H, int S, long rows,
                          Strides4 dos, Strides4 osr) {
  constexpr int LANES = D / 8;
  const long row = (long)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  if (row >= rows) return;             // whole groups of lanes
  const int d = threadIdx.x % LANES * 8;
  const int s = (int)(row % S);
  const int h = (int)((row / S) % H);
  const long b = row / ((long)S * H);
  typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
  const uint4_t dv = *(const uint4_t*)(dout + b * dos.sb + h * dos.sh + s * dos.ss + d);
  const uint4_t ov = *(const uint4_t*)(o + b * osr.sb + h * osr.sh + s * osr.ss + d);
  float acc = 0.f;
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    union { unsigned i; float f; } dl, dh, ol, oh;
    dl.i = dv[j] << 16; dh.i = dv[j] & 0xffff0000u;
    ol.i = ov[j] << 16; oh.i = ov[j] & 0xffff0000u;
    acc = fmaf(dl.f, ol.f, acc);
    acc = fmaf(dh.f, oh.f, acc);
  }
  #pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (d == 0) delta[row] = acc - (dlse ? dlse[row] : 0.f);
}

template <int D>
__global__ void __launch_bounds__(256, D == 64 ? 4 : 2)
attn_bwd_dq_kernel(const short* __restrict__ dout, const short* __restrict__ q,
                   const short* __restrict__ k, const short* __restrict__ v,
                   const float* __restrict__ lse,
                   const float* __restrict__ delta, short* __restrict__ dq,
                   int B, int H, int Hkv, int S, float scale, int causal,
                   int nbx, Strides4 dos, Strides4 qs, Strides4 ks, Strides4 vs,
                   Strides4 dqs) {
  constexpr int NSL = D / 16;
  constexpr int NDT = D / 32;
  __shared__ __attribute__((aligned(16))) short k0[64 * D], k1[64 * D];
  __shared__ __attribute__((aligned(16))) short v0[64 * D], v1[64 * D];

  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63;
  const int half = l >> 5;
  const Image<D> image(l);

  int bx, b, h;
  head_tile_map(nbx, B, H, Hkv, &bx, &b, &h);
  if (causal) bx = nbx - 1 - bx;   // those that see most keys start first
  const int hk = h / (H / Hkv);
  const int w0 = bx * ROWS + 32 * wid;      // this wave's first row
  const int row = w0 + (l & 31), rowc = min(row, S - 1);

  const long stat = ((long)b * H + h) * S + rowc;
  const float my_lse2 = lse[stat] * LOG2E, my_delta = delta[stat];
  const float scale2 = scale * LOG2E;
  bf16x8_t qf[NSL], dof[NSL];
  {
    const short* qr = q + (long)b * qs.sb + (long)h * qs.sh + (long)rowc * qs.ss + 8 * half;
    const short* dr = dout + (long)b * dos.sb + (long)h * dos.sh + (long)rowc * dos.ss + 8 * half;
    #pragma unroll
    for (int s = 0; s < NSL; ++s) {
      qf[s] = *(const bf16x8_t*)(qr + 16 * s);
      dof[s] = *(const bf16x8_t*)(dr + 16 * s);
    }
  }
  const short* kh = k + (long)b * ks.sb + (long)hk * ks.sh;
  const short* vh = v + (long)b * vs.sb + (long)hk * vs.sh;
  const unsigned ka = copy_at<D>(ks.ss), va = copy_at<D>(vs.ss);

  f32x16_t acc[NDT];
  #pragma unroll
  for (int t = 0; t < NDT; ++t) acc[t] = {};

  const int end = causal ? min(S, bx * ROWS + ROWS) : S;
  auto tile = [&](auto odd, int c0) INLINE {
    constexpr bool O = decltype(odd)::value;
    if (c0 + 64 < end) {
      copy_rows<D>(O ? k0 : k1, kh, ks.ss, ka, c0 + 64, S, wid);
      copy_rows<D>(O ? v0 : v1, vh, vs.ss, va, c0 + 64, S, wid);
    }
    const short* kimg = O ? k1 : k0;
    const short* vimg = O ? v1 : v0;
    #pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int cs = c0 + 32 * sub;
      if (cs >= S || (causal && cs > w0 + 31)) continue;
      const Image<D> at = image.again();
      f32x16_t sacc = {}, dp = {};
      #pragma unroll
      for (int s = 0; s < NSL; ++s) {
        sacc = mma(at.row(kimg, sub, s), qf[s], sacc);
        dp = mma(at.row(vimg, sub, s), dof[s], dp);
      }
      #pragma unroll
      for (int r = 0; r < 16; ++r) {
        #pragma clang fp contract(off)
        sacc[r] = __builtin_amdgcn_exp2f(sacc[r] * scale2 - my_lse2);
      }
      if (cs + 31 >= S || (causal && cs + 31 > w0)) {
        asm volatile("");      // a branch, not 16 selects in every tile
        const int seen = (causal ? min(S, row + 1) : S) - cs - 4 * half;
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          if ((r & 3) + 8 * (r >> 2) >= seen) sacc[r] = 0.f;
      }
      #pragma unroll
      for (int r = 0; r < 16; ++r) sacc[r] = sacc[r] * (dp[r] - my_delta) * scale;
      bf16x8_t ds[2];
      pack_frags(sacc, ds);
      #pragma unroll
      for (int t = 0; t < NDT; ++t)
        #pragma unroll
        for (int s = 0; s < 2; ++s) acc[t] = mma(at.col(kimg, sub, t, s), ds[s], acc[t]);
    }
    next_tile();
  };
  copy_rows<D>(k0, kh, ks.ss, ka, 0, S, wid);
  copy_rows<D>(v0, vh, vs.ss, va, 0, S, wid);
  next_tile();
  for (int c0 = 0; c0 < end; c0 += 128) {
    tile(std::false_type{}, c0);
    if (c0 + 64 < end) tile(std::true_type{}, c0 + 64);
  }

  if (row < S) {
    short* to = dq + (long)b * dqs.sb + (long)h * dqs.sh + (long)row * dqs.ss + 4 * half;
    #pragma unroll
    for (int t = 0; t < NDT; ++t)
      #pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        bf16x4 pk;
        #pragma unroll
        for (int j = 0; j < 4; ++j) pk[j] = f2bf(acc[t][rq * 4 + j]);
        *(bf16x4*)(to + 32 * t + 8 * rq) = pk;
      }
  }
}

template <int D>
__global__ void __launch_bounds__(256, D == 64 ? 3 : 1)
attn_bwd_dkv_kernel(const short* __restrict__ dout, const short* __restrict__ q,
                    const short* __restrict__ k, const short* __restrict__ v,
                    const float* __restrict__ lse,
                    const float* __restrict__ delta, short* __restrict__ dk,
                    short* __restrict__ dv, int B, int H, int Hkv, int S,
                    float scale, int causal, int nbx, Strides4 dos, Strides4 qs,
                    Strides4 ks, Strides4 vs, Strides4 dks, Strides4 dvs) {
  constexpr int NSL = D / 16;
  constexpr int NDT = D / 32;
  constexpr bool ALONE = D == 128;     // one wave to a SIMD
  __shared__ __attribute__((aligned(16))) short q0[64 * D], q1[64 * D];
  __shared__ __attribute__((aligned(16))) short d0[64 * D], d1[64 * D];
  // of a tile's rows: logsumexp in base 2, then delta
  __shared__ __attribute__((aligned(16))) float s0[128], s1[128];

  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int lk = l & 31;
  const int half = l >> 5;
  const Image<D> image(l);

  int bx, b, hk;
  head_tile_map(nbx, B, Hkv, Hkv, &bx, &b, &hk);   // the first are the longest
  const int group = H / Hkv;
  const int w0 = bx * ROWS + 32 * wid;      // this wave's first row
  const int row = w0 + lk, rowc = min(row, S - 1);
  const float scale2 = scale * LOG2E;

  bf16x8_t kf[NSL], vf[NSL];
  {
    const short* kr = k + (long)b * ks.sb + (long)hk * ks.sh + (long)rowc * ks.ss + 8 * half;
    const short* vr = v + (long)b * vs.sb + (long)hk * vs.sh + (long)rowc * vs.ss + 8 * half;
    #pragma unroll
    for (int s = 0; s < NSL; ++s) {
      kf[s] = *(const bf16x8_t*)(kr + 16 * s);
      vf[s] = *(const bf16x8_t*)(vr + 16 * s);
    }
  }
  const unsigned qa = copy_at<D>(qs.ss), da = copy_at<D>(dos.ss);

  f32x16_t dvacc[NDT], dkacc[NDT];
  #pragma unroll
  for (int t = 0; t < NDT; ++t) { dvacc[t] = {}; dkacc[t] = {}; }

  // Tiles c0, c0 + 64 ... of one head after the other.  Row statistics are
  // fetched before a tile's copies, behind which they would wait, and put down
  // at the end of the tile.
  const int first = causal ? bx * ROWS : 0;
  float stat = 0.f;
  auto fetch = [&](int g, int c0) INLINE {
    if (tid >= 128) return;
    const long r = ((long)b * H + hk * group + g) * S + min(c0 + l, S - 1);
    stat = (tid < 64 ? lse : delta)[r];
  };
  auto put = [&](float* to) INLINE {
    if (tid < 128) to[tid] = tid < 64 ? stat * LOG2E : stat;
  };
  auto copy = [&](short* qi, short* di, int g, int c0) INLINE {
    const int h = hk * group + g;
    copy_rows<D>(qi, q + (long)b * qs.sb + (long)h * qs.sh, qs.ss, qa, c0, S, wid);
    copy_rows<D>(di, dout + (long)b * dos.sb + (long)h * dos.sh, dos.ss, da, c0, S, wid);
  };
  int g = 0, c0 = first;
  auto tile = [&](auto odd) INLINE {
    constexpr bool O = decltype(odd)::value;
    const bool turn = c0 + 64 >= S;
    const int gn = turn ? g + 1 : g, cn = turn ? first : c0 + 64;
    if (gn < group) {
      fetch(gn, cn);
      copy(O ? q0 : q1, O ? d0 : d1, gn, cn);
    }
    const short* qimg = O ? q1 : q0;
    const short* dimg = O ? d1 : d0;
    Image<D> at = image.again();
    f32x16_t sacc[2], dp[2];
    bf16x8_t p[2][2], ds[2][2];
    auto scores = [&](int sub) INLINE {
      sacc[sub] = {};
      dp[sub] = {};
      #pragma unroll
      for (int s = 0; s < NSL; ++s) {
        sacc[sub] = mma(at.row(qimg, sub, s), kf[s], sacc[sub]);
        dp[sub] = mma(at.row(dimg, sub, s), vf[s], dp[sub]);
      }
    };
    auto weights = [&](int sub, bool edge) INLINE {
      const int cs = c0 + 32 * sub;
      const float* stats = (O ? s1 : s0) + 32 * sub + 4 * half;
      #pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const f32x4 lse4 = *(const f32x4*)(stats + 8 * rq);
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = sacc[sub][4 * rq + j] * scale2;
          sacc[sub][4 * rq + j] = __builtin_amdgcn_exp2f(x - lse4[j]);
        }
      }
      if (edge) {
        const int lo = causal ? row - cs - 4 * half : -4, hi = S - cs - 4 * half;
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = (r & 3) + 8 * (r >> 2);
          if (i < lo || i >= hi) sacc[sub][r] = 0.f;
        }
      }
      pack_frags(sacc[sub], p[sub]);
      #pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const f32x4 del4 = *(const f32x4*)(stats + 64 + 8 * rq);
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 4 * rq + j;
          dp[sub][r] = sacc[sub][r] * (dp[sub][r] - del4[j]) * scale;
        }
      }
      pack_frags(dp[sub], ds[sub]);
    };
    auto sums = [&](int sub) INLINE {
      #pragma unroll
      for (int t = 0; t < NDT; ++t)
        #pragma unroll
        for (int s = 0; s < 2; ++s) {
          dvacc[t] = mma(p[sub][s], at.col(dimg, sub, t, s), dvacc[t]);
          dkacc[t] = mma(ds[sub][s], at.col(qimg, sub, t, s), dkacc[t]);
        }
    };
    const bool edge = c0 + 64 > S || (causal && w0 + 31 > c0);
    if (ALONE && !edge) {
      // The products in the order that they run in, each with the LDS read of
      // an operand AHEAD of it and, two behind the scores that it takes, one
      // score's weight.
      constexpr int N = 2 * NSL, M = 4 * NDT, AHEAD = 6, LAG = 2;
      auto operand = [&](auto n) INLINE {
        constexpr int I = decltype(n)::value, J = I - 2 * N;
        if constexpr (J < 0) return at.row(I & 1 ? dimg : qimg, I / N, I % N / 2);
        else return at.col(J & 1 ? qimg : dimg, J / M, J % M / 4, J / 2 & 1);
      };
      auto product = [&](auto n, bf16x8_t x) INLINE {
        constexpr int I = decltype(n)::value, J = I - 2 * N;
        if constexpr (J < 0) {
          constexpr int U = I / N, T = I % N / 2;
          if constexpr (I & 1) dp[U] = mma(x, vf[T], T == 0 ? f32x16_t{} : dp[U]);
          else sacc[U] = mma(x, kf[T], T == 0 ? f32x16_t{} : sacc[U]);
        } else {
          constexpr int U = J / M, T = J % M / 4, H = J / 2 & 1;
          if constexpr (J & 1) dkacc[T] = mma(ds[U][H], x, dkacc[T]);
          else dvacc[T] = mma(p[U][H], x, dvacc[T]);
        }
      };
      f32x4 ls[4], de[4];
      unsigned pw[8], dw[8];
      float sx[16], dx[16];
      auto stats = [&](int sub, auto n) INLINE {
        constexpr int I = decltype(n)::value;
        const float* from = (O ? s1 : s0) + 32 * sub + 4 * half + 8 * I;
        ls[I] = *(const f32x4*)from;
        de[I] = *(const f32x4*)(from + 64);
      };
      auto weight = [&](auto n) INLINE {
        constexpr int I = decltype(n)::value, U = I / 16, R = I % 16;
        const float x = sx[R] * scale2;
        const float e = __builtin_amdgcn_exp2f(x - ls[R / 4][R % 4]);
        sx[R] = e;
        dx[R] = e * (dx[R] - de[R / 4][R % 4]) * scale;
        if constexpr (R & 1) {
          pw[R / 2] = cvt_pk_bf16(sx[R - 1], e);
          dw[R / 2] = cvt_pk_bf16(dx[R - 1], dx[R]);
        }
        if constexpr (R % 8 == 7) {
          p[U][R / 8] = exchange(pw + R / 8 * 4);
          ds[U][R / 8] = exchange(dw + R / 8 * 4);
        }
      };
      static_assert(!ALONE || (N == 16 && M == 16), "a score to a product");
      bf16x8_t ring[AHEAD];
      each<AHEAD>([&](auto n) INLINE { ring[n] = operand(n); });
      each<2 * (N + M)>([&](auto n) INLINE {
        constexpr int I = decltype(n)::value, R = I - N - LAG;
        product(n, ring[I % AHEAD]);
        if constexpr (I + AHEAD < 2 * (N + M))
          ring[I % AHEAD] = operand(std::integral_constant<int, I + AHEAD>{});
        if constexpr (I > N && I <= 2 * N + 4 && (I - 1) % N < 4) {
          #pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int at = (I - 1) % N * 4 + r;
            sx[at] = sacc[(I - 1) / N - 1][at];
            dx[at] = dp[(I - 1) / N - 1][at];
            asm volatile("" : "+v"(sx[at]), "+v"(dx[at]));
          }
        }
        if constexpr (R >= 0 && R < 32) weight(std::integral_constant<int, R>{});
        if constexpr (I < 4) stats(0, n);
        else if constexpr (R >= 0 && R < 16 && R % 4 == 3)
          stats(1, std::integral_constant<int, R / 4>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      #pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int cs = c0 + 32 * sub;
        if (cs >= S || (causal && cs + 31 < w0)) continue;
        at = image.again();
        scores(sub);
        weights(sub, edge);
        sums(sub);
      }
    }
    put(O ? s0 : s1);
    g = gn;
    c0 = cn;
    next_tile();
  };
  fetch(0, first);
  copy(q0, d0, 0, first);
  put(s0);
  next_tile();
  while (g < group) {
    tile(std::false_type{});
    if (g < group) tile(std::true_type{});
  }

  // a lane has a column, its registers rows
  #pragma unroll
  for (int t = 0; t < NDT; ++t)
    #pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int kg = w0 + (r & 3) + 8 * (r >> 2) + 4 * half;
      if (kg < S) {
        dk[(long)b * dks.sb + (long)hk * dks.sh + (long)kg * dks.ss + 32 * t + lk]
            = f2bf(dkacc[t][r]);
        dv[(long)b * dvs.sb + (long)hk * dvs.sh + (long)kg * dvs.ss + 32 * t + lk]
            = f2bf(dvacc[t][r]);
      }
    }
}

// A lane's place in a tile of 64 rows is a 32-bit offset: views whose rows lie
// farther apart than that allows are copied.
torch::Tensor near_rows(const torch::Tensor& t) {
  return t.stride(2) < (1l << 24) ? t : t.contiguous();
}

template <int D>
void launch(const torch::Tensor& dout, const torch::Tensor& q,
            const torch::Tensor& k, const torch::Tensor& v,
            const torch::Tensor& o, const torch::Tensor& lse,
            const torch::Tensor& delta, const torch::Tensor& dq,
            const torch::Tensor& dk, const torch::Tensor& dv, int B, int H,
            int Hkv, int S, float scale, bool causal, const float* dlse) {
  auto st = scaffold_stream();
  const long rows = (long)B * H * S, per = 256 / (D / 8);
  const int nbx = (S + ROWS - 1) / ROWS;
  const short *dop = (const short*)dout.data_ptr(), *qp = (const short*)q.data_ptr(),
              *kp = (const short*)k.data_ptr(), *vp = (const short*)v.data_ptr();
  const float* lsep = lse.data_ptr<float>();
  float* dp = delta.data_ptr<float>();
  const Strides4 dos = strides_of(dout), qs = strides_of(q), ks = strides_of(k),
                 vs = strides_of(v);
  hipLaunchKernelGGL((attn_delta_strided_kernel<D>), dim3((unsigned)((rows + per - 1) / per)),
                     dim3(256), 0, st, dop, (const short*)o.data_ptr(), dlse, dp, H, S,
                     rows, dos, strides_of(o));
  hipLaunchKernelGGL((attn_bwd_dq_kernel<D>), dim3(nbx * B * H), dim3(256), 0, st, dop,
                     qp, kp, vp, lsep, dp, (short*)dq.data_ptr(), B, H, Hkv, S, scale,
                     causal ? 1 : 0, nbx, dos, qs, ks, vs, strides_of(dq));
  hipLaunchKernelGGL((attn_bwd_dkv_kernel<D>), dim3(nbx * B * Hkv), dim3(256), 0, st,
                     dop, qp, kp, vp, lsep, dp, (short*)dk.data_ptr(),
                     (short*)dv.data_ptr(), B, H, Hkv, S, scale, causal ? 1 : 0, nbx,
                     dos, qs, ks, vs, strides_of(dk), strides_of(dv));
  HIP_CHECK(hipGetLastError());
}

}  // namespace

void attn_bwd_mfma(torch::Tensor dout, torch::Tensor q, torch::Tensor k,
                   torch::Tensor v, torch::Tensor o, torch::Tensor lse,
                   torch::Tensor delta, torch::Tensor dq, torch::Tensor dk,
                   torch::Tensor dv, int B, int H, int Hkv, int S, int D,
                   double scale, bool causal, const float* dlse_ptr) {
  dout = near_rows(dout);
  q = near_rows(q);
  k = near_rows(k);
  v = near_rows(v);
  if (D == 64)
    launch<64>(dout, q, k, v, o, lse, delta, dq, dk, dv, B, H, Hkv, S, (float)scale, causal, dlse_ptr);
  else if (D == 128)
    launch<128>(dout, q, k, v, o, lse, delta, dq, dk, dv, B, H, Hkv, S, (float)scale, causal, dlse_ptr);
  else TORCH_CHECK(false, "attn_bwd_mfma: unsupported D ", D);
}
