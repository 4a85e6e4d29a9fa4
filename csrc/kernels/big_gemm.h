// Products of large matrices, bf16 operands and float32 sums: y = x w^T, the gradients
// dx = dy w and dW = dy^T x.  One kernel, whose operands lie with the summed index along
// their rows or down them.
//
// What bounds it: a compute unit's products of 256 x 256 x 64 take 2048 cycles, its copies
// of 64 KB into LDS 1500 and its reads from LDS 1000 beside them, and the card's power, which
// lowers the clock to 1.7 GHz where the matrix cores are busy for 84 % of the time.
//
//  * 4 waves, one to a SIMD, of 128 x 128 outputs: with 8 waves of 128 x 64 the reads from
//    LDS are half as many again, and tiles of 128 take twice the copies.  The sums fill all
//    256 accumulator registers of a wave.
//  * Two stages of 64 of the summed index in LDS, copied as whole lines of 128 bytes.  (Four
//    of 32, with half lines, are a quarter slower.)  Reads are half a stage ahead of the
//    products, copies up to two; all of them lie spread between the products.
//  * A block goes from tile to tile, and the next tile's copies and reads begin during
//    the last stage of the one before.
//  * Results are stored by 16 lanes with 256 bytes of a row: in pieces of 64 bytes, as the
//    products leave them, a unit writes 27 bytes a ns instead of 72.  x w^T has w's rows
//    spread over the products, so that a lane's outputs are neighbours; the gradients'
//    go through LDS.
//
// In us, a library and this, operands out of memory: x w^T, 16384 x 2304 x 768 71 and 51,
// 16384 x 3072 x 768 78 and 67, 8192^3 693 and 720; dx, 16384 x 3072 x 768 87 and 68, 8192 x
// 14336 x 4096 721 and 631 (1525 TF/s); dW, 28672 x 4096 x 8192 1654 and 1271 (1514 TF/s),
// 4096 x 4096 x 8192 241 and 186.
#pragma once

#include "../device.h"

struct BigArgs {
  const short *a, *b;            // operands, of rows of lda and ldb
  const short* bias;             // (N) or null; x w^T only
  const short* res;              // (M, N) of rows of ldy, added to the result
  short* y;                      // (M, N) of rows of ldy
  long lda, ldb, ldy;
  int M, N, K;
  int am, bn;                    // of a and of b that there are to read, M and N or more or less
  unsigned tiles;
  bool stream;                   // the result goes past the caches
};

// a residual is added before the result is rounded, or to the rounded result
enum BigAct { BIG_NONE, BIG_GELU_ERF, BIG_RESIDUAL, BIG_RESIDUAL_LAST };

namespace big {

// y(m, n) = sum over k of A(m, k) B(n, k).  An operand lies with k along its rows (m, k),
// or, COL, with k down (k, m).
//
// 4 waves, one to a SIMD, of 128 x 16 NT outputs.  Stages of 64 of k, two in LDS.
template <bool ACOL, bool BCOL, int NT, int ACT>
__global__ void __launch_bounds__(256, 1)
gemm_kernel(BigArgs a) {
  constexpr int MT = 8, BM = 32 * MT, BN = 32 * NT, BK = 64;
  constexpr int CA = BM / 32, CB = BN / 32, C = CA + CB;           // copies of a wave
  constexpr int RA = ACOL ? 2 * MT : MT, RB = BCOL ? 2 * NT : NT, R = RA + RB;
  constexpr int Q1 = MT * NT;                                      // products of half a stage
  __shared__ __attribute__((aligned(16))) short a0[BM * BK], b0[BN * BK];
  __shared__ __attribute__((aligned(16))) short a1[BM * BK], b1[BN * BK];
  constexpr int TURN = 16 * NT + 8;                                // row of the turned result
  __shared__ __attribute__((aligned(16))) short turned[BCOL ? 4 * 16 * TURN : 8];

  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int lr = l & 15, lg = l >> 4, wm = wid >> 1, wn = wid & 1;
  const int ns = (a.K + 2 * BK - 1) / (2 * BK) * 2;                // an even number
  const unsigned gm = (a.M + BM - 1) / BM, gn = (a.N + BN - 1) / BN;

  // A lane's places in its wave's copies.  k along the rows: 8 rows of 8 chunks, chunk c of a
  // row at c ^ (row / 2 % 8), so that the 16 rows of a read lie in different banks; of B, row
  // j of a wave's 16 NT is j % 16 * NT + j / 16, so that a lane's outputs are neighbours.
  // k down: units of 4 x 32, whose halves change places where k / 8 is odd.
  auto along = [&](int i, long ld, bool spread) INLINE {
    const int row = (i * 4 + wid) * 8 + (l >> 3);
    const int in = row % (16 * NT), at = spread ? row - in + (in & 15) * NT + (in >> 4) : row;
    return 2 * ((unsigned)at * (unsigned)ld + 8 * ((l & 7) ^ (row >> 1 & 7)));
  };
  auto down = [&](int i, long ld, int units) INLINE {
    const int s = (i * 4 + wid) * 64 + l, quad = (s >> 4) / units;
    const int col = (s >> 4) % units * 32 + ((s >> 1 ^ quad >> 1) & 1) * 16 + (s & 1) * 8;
    return 2 * ((unsigned)(quad * 4 + (s >> 2 & 3)) * (unsigned)ld + col);
  };
  unsigned pa[CA], pb[CB];
  #pragma unroll
  for (int i = 0; i < CA; ++i) pa[i] = ACOL ? down(i, a.lda, MT) : along(i, a.lda, false);
  #pragma unroll
  for (int i = 0; i < CB; ++i) pb[i] = BCOL ? down(i, a.ldb, NT) : along(i, a.ldb, true);

  // tile t: 8 down, then across
  auto place = [&](unsigned t, int& m0, int& n0) INLINE {
    const unsigned group = t / (8 * gn), high = min(8u, gm - 8 * group);
    const unsigned in = t - group * 8 * gn;
    m0 = (int)(8 * group + in % high) * BM;
    n0 = (int)(in / high) * BN;
  };
  // this block's tiles: every gridDim.x-th from id on; an XCD's lie next to each other
  const unsigned G = gridDim.x, q8 = G / 8, r8 = G % 8, xcd = blockIdx.x % 8;
  const unsigned id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) +
                      blockIdx.x / 8;

  // what is copied next: a tile, its stage, and where in memory that begins.  What lies
  // behind the operand's end, size elements on, reads as zero.
  struct Place { unsigned long at; unsigned size; };
  unsigned tc = id;
  int sc = 0, mc, nc;
  Place ca, cb;
  auto where = [&](auto col, const short* from, long ld, int first, int end) INLINE {
    const int k = sc * BK;
    long at, size;
    if (decltype(col)::value) {
      const int rows = min(BK, a.K - k);
      at = (long)min(k, a.K) * ld + first;
      size = rows > 0 ? (rows - 1) * ld + end - first : 0;
    } else {
      at = (long)first * ld + k;
      size = (min(256, end - first) - 1) * ld + BK;
    }
    return Place{(unsigned long)(from + at), (unsigned)(2 * size)};
  };
  auto seek = [&]() INLINE {
    ca = where(std::integral_constant<bool, ACOL>{}, a.a, a.lda, mc, a.am);
    cb = where(std::integral_constant<bool, BCOL>{}, a.b, a.ldb, nc, a.bn);
  };
  place(tc, mc, nc);
  seek();
  auto copy = [&](short* to, const Place& from, unsigned off, int i) INLINE {
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((unsigned long)same((unsigned)(from.at >> 32)) << 32 | same((unsigned)from.at)),
        0, (int)same(from.size), 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (__attribute__((address_space(3))) void*)(to + (i * 4 + wid) * 512), 16, off, 0, 0,
        0);
  };
  using std::integral_constant;
  auto stage = [&](auto odd, auto j) INLINE {
    constexpr int J = decltype(j)::value;
    constexpr bool O = decltype(odd)::value;
    if constexpr (J < CB) copy(O ? b1 : b0, cb, pb[J], J);
    else copy(O ? a1 : a0, ca, pa[J - CB], J - CB);
  };
  auto advance = [&]() INLINE {
    if (++sc == ns) {
      sc = 0;
      // behind the last tile this block's first once more, which nothing takes
      tc = tc + G < a.tiles ? tc + G : id;
      place(tc, mc, nc);
    }
    seek();
  };

  // reads
  const int arow = ACOL ? 0 : (wm * 16 * MT + lr) * BK, brow = BCOL ? 0 : (wn * 16 * NT + lr) * BK;
  const int chunk[2] = {8 * (lg ^ (lr >> 1 & 7)), 8 * ((4 + lg) ^ (lr >> 1 & 7))};
  // k down: this lane's 8 bytes of an even or odd sixteen of columns
  const int in4 = (lr >> 2) * 32 + (lr & 3) * 4;
  const int even = in4 + (lg & 1) * 16, odd16 = in4 + (1 - (lg & 1)) * 16;
  typedef __attribute__((address_space(3))) bf16x4* P4;
  // sixteen f of those from unit `first` on, quad q of a lane's two of half p
  auto quad = [&](const short* img, int units, int first, int f, int p, int q) INLINE {
    const int at = ((8 * p + 2 * lg + q) * units + first + f / 2) * 128;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((P4)(img + at + (f & 1 ? odd16 : even)));
  };
  f32x4 acc[MT][NT];
  union Frag { bf16x8 v; bf16x4 q[2]; };
  Frag fa[2][MT], fb[2][NT];
  auto read = [&](auto half, auto odd, auto r) INLINE {
    constexpr int P = decltype(half)::value, N = decltype(r)::value;
    constexpr bool O = decltype(odd)::value;
    const short *ai = O ? a1 : a0, *bi = O ? b1 : b0;
    if constexpr (N < RB) {
      if constexpr (BCOL) {
        fb[P][N / 2].q[N % 2] = quad(bi, NT, wn * (NT / 2), N / 2, P, N % 2);
      } else {
        fb[P][N].v = *(const bf16x8*)(bi + brow + 16 * N * BK + chunk[P]);
      }
    } else {
      if constexpr (ACOL) {
        constexpr int X = N - RB;
        fa[P][X / 2].q[X % 2] = quad(ai, MT, wm * (MT / 2), X / 2, P, X % 2);
      } else {
        fa[P][N - RB].v = *(const bf16x8*)(ai + arow + 16 * (N - RB) * BK + chunk[P]);
      }
    }
  };

  // One stage out of registers, a half after the other.  Its second half is read from LDS
  // beside the first products; then (FREE) all waves have what they need of its place, and
  // the copies of the stage after the next go there; when (HERE) the next stage has come,
  // in all waves, its first half is read.
  constexpr int READ1 = R <= 16 || R == 24 ? 2 : 1, READ2 = READ1;
  constexpr int FREE = READ1 * (R - 1) + (R > 24 ? 6 : R == 24 ? 4 : 2);
  constexpr int COPY = NT == 8 ? 5 : 4;
  constexpr int HERE = NT < 8 ? 56 : R > 24 ? 84 : R == 24 ? 64 : 88;
  static_assert(FREE + 1 + COPY * (C - 1) < 2 * Q1 && HERE + 1 + READ2 * (R - 1) < 2 * Q1 &&
                HERE + 1 >= Q1, "schedule");
  // stores of a tile, of which the first stage behind it takes no notice
  constexpr int STORES = BCOL ? MT * NT / 2 : 4 * MT;
  auto step = [&](auto odd, auto first) INLINE {
    constexpr bool O = decltype(odd)::value, F = decltype(first)::value;
    constexpr integral_constant<bool, O> this_;
    constexpr integral_constant<bool, !O> other;
    each<2 * Q1>([&](auto q) INLINE {
      constexpr int Q = decltype(q)::value, P = Q / Q1, I = Q % Q1 / NT, T = Q % NT;
      // In assembly: the builtin's sums, which fill all accumulator registers, the compiler
      // moves about, 900 times a tile.  Operands come from LDS alone, so that none is the
      // result of a vector instruction two wait states before, which would have to be
      // waited for (tests/unit/test_big_gemm_asm.py); waits before each are 5 to 8 % of the
      // time.
      const bf16x8 x = BCOL ? fb[P][T].v : fa[P][I].v, w = BCOL ? fa[P][I].v : fb[P][T].v;
      if constexpr (F && P == 0)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                     : "=a"(acc[I][T]) : "v"(x), "v"(w));
      else
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[I][T]) : "v"(x), "v"(w));
      if constexpr (Q % READ1 == 0 && Q / READ1 < R)
        read(integral_constant<int, 1>{}, this_, integral_constant<int, Q / READ1>{});
      if constexpr (Q == FREE) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);                        // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (Q > FREE && (Q - FREE - 1) % COPY == 0 && (Q - FREE - 1) / COPY < C)
        stage(this_, integral_constant<int, (Q - FREE - 1) / COPY>{});
      if constexpr (Q == HERE) {
        constexpr int asked = std::min((HERE - FREE - 1 + COPY) / COPY, C);
        constexpr int vm = std::min(63, asked + (F ? STORES : 0));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0f70 | (vm & 15) | (vm >> 4) << 14);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (Q > HERE && (Q - HERE - 1) % READ2 == 0 && (Q - HERE - 1) / READ2 < R)
        read(integral_constant<int, 0>{}, other, integral_constant<int, (Q - HERE - 1) / READ2>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    advance();
  };
  constexpr std::true_type yes;
  constexpr std::false_type no;
  each<C>([&](auto j) INLINE { stage(no, j); });
  advance();
  each<C>([&](auto j) INLINE { stage(yes, j); });
  advance();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70);                              // vmcnt(0): step() counts stores
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  each<R>([&](auto r) INLINE { read(integral_constant<int, 0>{}, no, r); });

  for (unsigned t = id; t < a.tiles; t += G) {
    step(no, yes);
    step(yes, no);
    for (int s = 2; s < ns; s += 2) {
      step(no, no);
      step(yes, no);
    }
    // The last products' results, which take up to 18 wait states.  Every sum goes through a
    // statement behind the wait, so that no read of it can be placed before that.
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    #pragma unroll
    for (int i = 0; i < MT; ++i)
      #pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j]));
    __builtin_amdgcn_sched_barrier(0);
    int m0, n0;
    place(t, m0, n0);
    m0 += wm * 16 * MT;
    n0 += wn * 16 * NT;
    // opaque, so that places are not made ahead of the loop, where no register is free
    int lane = l;
    asm volatile("" : "+v"(lane));
    const int lr = lane & 15, lg = lane >> 4;
    // Sixteen rows from m on of the result (or what is added to it) as a buffer: what lies
    // behind the last row is not stored, but counts as a store, as step() has it.  A lane's
    // place is its row and column; one behind the last column lies outside of all.
    auto rows = [&](const short* y, int m) INLINE {
      const unsigned long at = (unsigned long)(y + (long)min(m, a.M - 1) * a.ldy + n0);
      const long size = m < a.M && n0 < a.N ? (min(16, a.M - m) - 1) * a.ldy + a.N - n0 : 0;
      return __builtin_amdgcn_make_buffer_rsrc(
          (void*)((unsigned long)same((unsigned)(at >> 32)) << 32 | same((unsigned)at)), 0,
          (int)same((unsigned)(2 * size)), 0x00020000);
    };
    auto at = [&](int row, int col) INLINE {
      return n0 + col < a.N ? 2 * (unsigned)(row * (int)a.ldy + col) : 0xfffffff0u;
    };
    auto act = [](float v) INLINE {
      return ACT == BIG_GELU_ERF ? gelu_erf(v) : v;
    };
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    auto store = [&](auto past) INLINE {
      constexpr int AUX = decltype(past)::value ? 2 : 0;           // not kept in the caches
      if constexpr (BCOL) {
        // a lane has four columns of each sixteen, of row lr: 16 rows at a time through LDS
        short* mine = turned + wid * 16 * TURN;
        #pragma unroll
        for (int i = 0; i < MT; ++i) {
          const auto to = rows(a.y, m0 + 16 * i);
          #pragma unroll
          for (int j = 0; j < NT; ++j)
            *(u32x2*)(mine + lr * TURN + 16 * j + 4 * lg) =
                u32x2{cvt_pk_bf16(acc[i][j][0], acc[i][j][1]), cvt_pk_bf16(acc[i][j][2], acc[i][j][3])};
          #pragma unroll
          for (int r = 0; r < NT / 2; ++r) {
            const int row = (64 * r + lane) / (2 * NT), col = (64 * r + lane) % (2 * NT) * 8;
            __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4*)(mine + row * TURN + col), to,
                                                   at(row, col), 0, AUX);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        // NT columns, which N is a multiple of, of four rows
        float b[NT] = {};
        if (a.bias)
          #pragma unroll
          for (int j = 0; j < NT; ++j) b[j] = bf2f(a.bias[min(n0 + lr * NT + j, a.N - 1)]);
        // the residual, asked for AHEAD stores before it is taken; 8 of 16 bytes do not fit
        // beside the next tile's operands
        constexpr int AHEAD = NT == 8 ? 5 : 7;
        constexpr bool RES = ACT == BIG_RESIDUAL || ACT == BIG_RESIDUAL_LAST;
        unsigned add[RES ? AHEAD + 1 : 1][NT / 2];
        auto ask = [&](int s) INLINE {
          const auto from = rows(a.res, m0 + s / 4 * 16);
          const unsigned place = at(4 * lg + s % 4, lr * NT);
          unsigned* to = add[s % (AHEAD + 1)];
          if constexpr (NT == 8) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(from, place, 0, 0);
            #pragma unroll
            for (int j = 0; j < 4; ++j) to[j] = v[j];
          } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(from, place, 0, 0);
            #pragma unroll
            for (int j = 0; j < 3; ++j) to[j] = v[j];
          }
        };
        if constexpr (RES)
          #pragma unroll
          for (int s = 0; s < AHEAD; ++s) ask(s);
        #pragma unroll
        for (int i = 0; i < MT; ++i) {
          const auto to = rows(a.y, m0 + 16 * i);
          #pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (RES)
              if (4 * i + r + AHEAD < 4 * MT) ask(4 * i + r + AHEAD);
            unsigned v[NT / 2];
            #pragma unroll
            for (int j = 0; j < NT / 2; ++j) {
              float lo = acc[i][2 * j][r] + b[2 * j], hi = acc[i][2 * j + 1][r] + b[2 * j + 1];
              if constexpr (ACT == BIG_RESIDUAL_LAST) {
                const unsigned y = cvt_pk_bf16(lo, hi);
                lo = __uint_as_float(y << 16);
                hi = __uint_as_float(y & 0xffff0000u);
              }
              if constexpr (RES) {
                lo += __uint_as_float(add[(4 * i + r) % (AHEAD + 1)][j] << 16);
                hi += __uint_as_float(add[(4 * i + r) % (AHEAD + 1)][j] & 0xffff0000u);
              }
              v[j] = cvt_pk_bf16(act(lo), act(hi));
            }
            const unsigned place = at(4 * lg + r, lr * NT);
            if constexpr (NT == 8)
              __builtin_amdgcn_raw_buffer_store_b128(u32x4{v[0], v[1], v[2], v[3]}, to, place, 0, AUX);
            else
              __builtin_amdgcn_raw_buffer_store_b96(u32x3{v[0], v[1], v[2]}, to, place, 0, AUX);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (a.stream) store(yes);
    else store(no);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);          // no copy is on its way into LDS at the end
}

}  // namespace big
