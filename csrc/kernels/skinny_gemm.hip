// y = x w^T for few rows x (a decode step: up to 64), bf16, float32 sums.
//
// What bounds it is reading w once, and with little of it the chain of a launch:
// an empty one takes 1.6 us, one that reads 24 KB a block and adds them up over 8
// waves 2.8.  A weight goes from memory to the one wave that multiplies it and
// nowhere else: a block has some rows of w, its 8 waves split the depth, and the
// rows of x, which every block reads, come out of the caches as the other operand
// of the 16x16x32 MFMA.  Each wave has the next span's loads in flight while it
// multiplies one, and what the end needs of bias and residual.  The waves' sums
// meet in LDS, where bias, residual, GELU or the gate's product join before the
// only rounding.

#include "../common.h"
#include "skinny.h"

namespace {

DEVINL f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  typedef __attribute__((ext_vector_type(8))) __bf16 v8;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

DEVINL float gelu_tanh(float z) {
  const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  // tanh(u) = 1 - 2 / (exp(2u) + 1), also at both ends
  return 0.5f * z * (2.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * u) + 1.f));
}

// sum over the lanes that are the same but for bit 4, or 5
DEVINL float pair_sum(float x, std::integral_constant<int, 16>) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
DEVINL float pair_sum(float x, std::integral_constant<int, 32>) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// and the lane N places on in its row of 16
template <int N> DEVINL float turn_sum(float x) {
  const int i = __builtin_bit_cast(int, x);
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                 0, i, 0x120 + N, 0xf, 0xf, true));
}

// waits for LDS alone: __syncthreads() would wait for weights on their way too
DEVINL void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// What a lane needs of bias and residual for 4 outputs, asked for when the
// kernel starts: behind the products each would be a wait of its own.  Where
// there is none, or it does not lie for it, any 8 bytes are, for a load in a
// branch is waited for where the ways meet.
struct Extra { bf16x4 bias, res; };

DEVINL Extra extra(const SkinnyArgs& a, int row, int n) {
  const bool b = a.bias && a.fours, r = a.res && a.fours;
  const int c = min(n, a.N - 4);
  return {*(const bf16x4*)((b ? a.bias : a.w) + (b ? c : 0)),
          *(const bf16x4*)((r ? a.res : a.w) + (r ? min(row, a.M - 1) * a.ldr + c : 0))};
}

// 4 outputs in a row of one row of x
template <int ACT>
DEVINL void put(const SkinnyArgs& a, const Extra& e, f32x4 s, int row, int n) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  short* y = a.y + row * a.ldy + n;
  if (a.fours) {
    const bf16x4 b = e.bias & (a.bias ? (short)-1 : (short)0);
    const bf16x4 r = e.res & (a.res ? (short)-1 : (short)0);
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] += bf2f(b[j]);
      if (ACT == SKINNY_GELU) s[j] = gelu_tanh(s[j]);
      s[j] += bf2f(r[j]);
    }
    *(u32x2*)y = u32x2{cvt_pk_bf16(s[0], s[1]), cvt_pk_bf16(s[2], s[3])};
    return;
  }
  #pragma unroll
  for (int j = 0; j < 4; ++j)
    if (n + j < a.N) {
      if (a.bias) s[j] += bf2f(a.bias[n + j]);
      if (ACT == SKINNY_GELU) s[j] = gelu_tanh(s[j]);
      if (a.res) s[j] += bf2f(a.res[row * a.ldr + n + j]);
      y[j] = (short)cvt_pk_bf16(s[j], s[j]);
    }
}

// MT tiles of 16 rows of x, RT tiles of rows of w (SWIGLU: half of them gate rows,
// half the up rows that go with them), NW waves.
//
// SEG: the 16 rows and columns of the matrix instruction are 16 / SEG rows of w
// and of x, each SEG times, at SEG places of the depth; of the products, those
// of equal places count.  So few rows of w make SEG times the blocks, which
// read a SEG-th each.
//
// S: the rows of x are normed first (layer norm with a bias, else RMS norm), by
// every block for itself: a wave has its share of the depth of all rows, S steps,
// in registers as the products take them, and only the sums go through LDS.
// Such a kernel is as long as its instructions in a row, 8 cycles each, and its
// waits.  768 to 2304, 1 row, 8 rows: rows normed by a wave each, rounded into LDS
// and read from there (11 KB of code), and bias asked for at the end 5.1 and 5.4 us;
// so 3.6 and 4.2; without the norm 3.1 and 3.4.
template <int MT, int RT, int NW, int ACT, int S, int SEG>
__global__ void __launch_bounds__(64 * NW)
skinny_kernel(SkinnyArgs a) {
  constexpr bool PAIR = ACT == SKINNY_SWIGLU;
  constexpr int U = MT + RT <= 3 ? 4 / SEG : SEG < 4 ? 2 : 1;
  constexpr int STEP = 32 * SEG;              // columns of a matrix instruction
  constexpr int SPAN = STEP * U;
  constexpr int OT = PAIR ? RT / 2 : RT;      // output tiles
  constexpr int R = 16 / SEG;                 // rows of one
  constexpr int TILES = (MT * OT + NW - 1) / NW;   // of a wave, at the end
  static_assert((SEG == 1 && !S) || (MT == 1 && NW == 8), "few rows");
  __shared__ __attribute__((aligned(16))) f32x4 part[NW][MT * RT][64];

  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int lr = l & 15, lg = l >> 4;
  const int n0 = blockIdx.x * R * OT;
  const int at = 8 * lg + 32 * (lr / R);      // of a step's columns, this lane's 8
  const short *wp[RT], *xp[MT];
  #pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int n = min(n0 + R * (r % OT) + lr % R, a.N - 1) + (r / OT) * a.N;
    wp[r] = a.w + (long)n * a.K + at;
  }
  #pragma unroll
  for (int m = 0; m < MT; ++m)
    xp[m] = a.x + (long)min(16 * m + lr % R, a.M - 1) * a.ldx + at;
  auto w_at = [&](int r, int c) { return *(const bf16x8*)(wp[r] + c); };
  auto x_at = [&](int m, int c) { return *(const bf16x8*)(xp[m] + c); };

  f32x4 acc[MT][RT];
  #pragma unroll
  for (int m = 0; m < MT; ++m)
    #pragma unroll
    for (int r = 0; r < RT; ++r) acc[m][r] = f32x4{0.f, 0.f, 0.f, 0.f};

  // where a lane's outputs are: of SEG^2 groups of lanes each has all of them
  const int orow = SEG == 1 ? lr : SEG == 2 ? l & 7 : l & 3;
  const int ocol = SEG == 1 ? 4 * lg : SEG == 2 ? (l >> 1) & 4 : 0;
  Extra ex[TILES];
  auto ask = [&] {
    #pragma unroll
    for (int i = 0; i < TILES; ++i) {
      const int t = min(wid + i * NW, MT * OT - 1);
      ex[i] = extra(a, 16 * (t / OT) + orow, n0 + R * (t % OT) + ocol);
    }
  };

  if constexpr (S) {
    __shared__ __attribute__((aligned(16))) float sums[2][R][NW];
    // Step i NW + wid of the depth; columns behind the end are read at its last
    // 8 and count as zero on both sides.  No load stands in a branch: the
    // compiler waits for all of them where two ways meet.
    const int last = (a.K - 1) / STEP * STEP;           // columns of the last step
    const int edge = min(at, a.K - 8 - last);
    auto col = [&](int i) { return (i * NW + wid) * STEP; };
    auto in = [&](int i) { return at < a.K - col(i); };
    auto from = [&](int i) {
      return min(col(i), last) + (col(i) < last ? 0 : edge - at);
    };
    bf16x8 x[S], w[RT][S], nw[S], nb[S];
    const short* nbp = a.nb ? a.nb : a.nw;
    auto fetch = [&](int i) {
      #pragma unroll
      for (int r = 0; r < RT; ++r) w[r][i] = w_at(r, from(i));
    };
    #pragma unroll
    for (int i = 0; i < S; ++i) x[i] = x_at(0, from(i));
    #pragma unroll
    for (int i = 0; i < S; ++i) fetch(i);
    #pragma unroll
    for (int i = 0; i < S; ++i) {
      nw[i] = *(const bf16x8*)(a.nw + at + from(i));
      nb[i] = *(const bf16x8*)(nbp + at + from(i));
    }
    ask();
    const float inv = 1.f / (float)a.K;
    // s: of the wave, by rows of x in 16 columns; to the whole depth's of this lane's row
    auto total = [&](float s, int n) {
      if constexpr (SEG == 2) s = turn_sum<8>(s);
      if constexpr (SEG == 4) s = turn_sum<8>(turn_sum<4>(s));
      if (l < R) sums[n][l][wid] = s;
      lds_barrier();
      const f32x4 lo = *(const f32x4*)&sums[n][lr % R][0];
      const f32x4 hi = *(const f32x4*)&sums[n][lr % R][4];
      return ((lo[0] + lo[1]) + (lo[2] + lo[3])) + ((hi[0] + hi[1]) + (hi[2] + hi[3]));
    };
    #pragma unroll
    for (int i = 0; i < S; ++i)
      if (col(i) >= last && !in(i)) x[i] = bf16x8{};
    auto normed = [&](auto layer) INLINE {
      constexpr bool LAYER = decltype(layer)::value;
      float mean = 0.f, s = 0.f;
      if constexpr (LAYER) {
        // the matrix instruction adds the rows up
        bf16x8 one;
        #pragma unroll
        for (int j = 0; j < 8; ++j) one[j] = 0x3f80;
        f32x4 t = {};
        #pragma unroll
        for (int i = 0; i < S; ++i) t = mma(one, x[i], t);
        mean = total(t[0], 0) * inv;
      }
      #pragma unroll
      for (int i = 0; i < S; ++i)
        if (!LAYER || col(i) < last || in(i))
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float d = bf2f(x[i][j]) - mean;
            s += d * d;
          }
      s = pair_sum(pair_sum(s, std::integral_constant<int, 16>{}),
                   std::integral_constant<int, 32>{});
      const float rstd = rsqrtf(total(s, 1) * inv + a.eps);
      #pragma unroll
      for (int i = 0; i < S; ++i) {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        u32x4 o;
        #pragma unroll
        for (int j = 0; j < 8; j += 2) {
          float y[2];
          #pragma unroll
          for (int k = 0; k < 2; ++k)
            y[k] = (bf2f(x[i][j + k]) - mean) * rstd * bf2f(nw[i][j + k]) +
                   (LAYER ? bf2f(nb[i][j + k]) : 0.f);
          o[j / 2] = cvt_pk_bf16(y[0], y[1]);
        }
        bf16x8 h = __builtin_bit_cast(bf16x8, o);
        if (col(i) >= last) {
          h = in(i) ? h : bf16x8{};
          #pragma unroll
          for (int r = 0; r < RT; ++r) w[r][i] = in(i) ? w[r][i] : bf16x8{};
        }
        #pragma unroll
        for (int r = 0; r < RT; ++r) acc[0][r] = mma(w[r][i], h, acc[0][r]);
      }
    };
    if (a.nb) normed(std::true_type{});
    else normed(std::false_type{});
  } else {
    struct Span { bf16x8 w[RT][U], x[MT][U]; };
    auto fetch = [&](Span& s, int k0) {
      #pragma unroll
      for (int u = 0; u < U; ++u) {
        #pragma unroll
        for (int r = 0; r < RT; ++r)
          s.w[r][u] = w_at(r, k0 + STEP * u);
        #pragma unroll
        for (int m = 0; m < MT; ++m) s.x[m][u] = x_at(m, k0 + STEP * u);
      }
    };
    auto use = [&](const Span& s) {
      #pragma unroll
      for (int u = 0; u < U; ++u)
        #pragma unroll
        for (int m = 0; m < MT; ++m)
          #pragma unroll
          for (int r = 0; r < RT; ++r) acc[m][r] = mma(s.w[r][u], s.x[m][u], acc[m][r]);
    };
    const int full = a.K / SPAN;               // whole spans
    Span s0, s1;
    int i = wid;
    if (i < full) fetch(s0, i * SPAN);
    ask();
    for (; i < full; i += 2 * NW) {
      if (i + NW < full) fetch(s1, (i + NW) * SPAN);
      use(s0);
      if (i + NW >= full) break;
      if (i + 2 * NW < full) fetch(s0, (i + 2 * NW) * SPAN);
      use(s1);
    }
    // what is left of the depth, a step at a time, by the waves that have had
    // one span less; columns behind the end are read at its last 8 and count
    // as zero on both sides
    const int left = (a.K - full * SPAN + STEP - 1) / STEP;
    const int mine = (wid - full % NW + NW) % NW;
    if (mine < left) {
      const int k0 = full * SPAN + STEP * mine;
      const bool in = k0 + at < a.K;
      const int c = in ? k0 : a.K - 8 - at;
      bf16x8 wv[RT], xv[MT];
      #pragma unroll
      for (int r = 0; r < RT; ++r) wv[r] = w_at(r, c);
      #pragma unroll
      for (int m = 0; m < MT; ++m) xv[m] = x_at(m, c);
      #pragma unroll
      for (int r = 0; r < RT; ++r) wv[r] = in ? wv[r] : bf16x8{};
      #pragma unroll
      for (int m = 0; m < MT; ++m) {
        xv[m] = in ? xv[m] : bf16x8{};
        #pragma unroll
        for (int r = 0; r < RT; ++r) acc[m][r] = mma(wv[r], xv[m], acc[m][r]);
      }
    }
  }
  #pragma unroll
  for (int m = 0; m < MT; ++m)
    #pragma unroll
    for (int r = 0; r < RT; ++r) part[wid][m * RT + r][l] = acc[m][r];
  __syncthreads();

  #pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int t = wid + i * NW;
    if (t >= MT * OT) break;
    const int m = t / OT, o = t % OT;
    // tile r's sums over waves, and over the places of the depth
    auto whole = [&](int r) {
      f32x4 s;
      if constexpr (SEG == 1) {
        s = part[0][r][l];
        #pragma unroll
        for (int v = 1; v < NW; ++v) s += part[v][r][l];
      } else if constexpr (SEG == 2) {
        // place c lies at lanes 16 (2 c + quad) + 8 c + row
        const int from = 16 * (ocol / 4) + orow;
        s = (part[2 * lg][r][from] + part[2 * lg][r][from + 40]) +
            (part[2 * lg + 1][r][from] + part[2 * lg + 1][r][from + 40]);
      } else {
        // at lanes 16 c + 4 c + row
        const int v = (l >> 2) & 7, from = (l >> 5) * 40 + orow;
        s = part[v][r][from] + part[v][r][from + 20];
        #pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = turn_sum<8>(turn_sum<4>(s[j]));
      }
      if constexpr (SEG > 1)
        #pragma unroll
        for (int j = 0; j < 4; ++j)
          s[j] = pair_sum(pair_sum(s[j], std::integral_constant<int, 16>{}),
                          std::integral_constant<int, 32>{});
      return s;
    };
    f32x4 s = whole(m * RT + o);
    if constexpr (PAIR) {
      const f32x4 up = whole(m * RT + OT + o);
      #pragma unroll
      for (int j = 0; j < 4; ++j) s[j] = s[j] / (1.f + __expf(-s[j])) * up[j];
    }
    const int row = 16 * m + orow, n = n0 + R * o + ocol;
    if (row < a.M && n < a.N && (SEG == 1 || l < 64 / (SEG * SEG)))
      put<ACT>(a, ex[i], s, row, n);
  }
}

template <int MT, int RT, int NW, int ACT, int S = 0, int SEG = 1>
void launch(const SkinnyArgs& a, hipStream_t st) {
  constexpr int OT = ACT == SKINNY_SWIGLU ? RT / 2 : RT, ROWS = 16 / SEG * OT;
  hipLaunchKernelGGL((skinny_kernel<MT, RT, NW, ACT, S, SEG>),
                     dim3((a.N + ROWS - 1) / ROWS), dim3(64 * NW), 0, st, a);
}

template <int RT, int ACT, int SEG>
void launch_norm(const SkinnyArgs& a, hipStream_t st) {
  const int steps = (a.K + 256 * SEG - 1) / (256 * SEG);
  if (steps == 1) launch<1, RT, 8, ACT, 1, SEG>(a, st);
  else if (steps == 2) launch<1, RT, 8, ACT, 2, SEG>(a, st);
  else if (steps == 3) launch<1, RT, 8, ACT, 3, SEG>(a, st);
  else launch<1, RT, 8, ACT, 4, SEG>(a, st);
}

// Up to 4 rows of x read w at four places of the depth at once, up to 8 at two: a
// load is whole lines of 128 bytes then (16 rows of w to a load have halves of
// 64), and x is read as often less.  A block has few rows of w as long as that
// fills the chip, and where as many blocks as 16 rows make would leave a last wave
// of them nearly empty.  In us, with 16 rows and more to a block, two waves of
// loads ahead (before), and now: 768 rows of w of 3072, 1 row of x 6.0 and 3.2, 8
// rows 7.1 and 5.1; 4096 of 4096, 1 row 9.3 and 8.0, 8 rows 10.0 and 9.1; 5120 of 4096,
// 2 rows 13.8 and 10.4, 5 rows 14.4 and 13.0; 128256 of 4096, 1 row 198 and 164, 8
// rows 205 and 182; pairs, 2 x 14336 of 4096, 1 row 52.0 and 41.2, 8 rows 49.9 and
// 44.6, 2 x 28672 of 8192 198 and 154, 197 and 161 (6.1 and 5.9 TB/s).  Many rows
// of w of little depth are as many short blocks: 50257 of 768, 1 row, 4 rows of w
// to a block 20.7, 8 15.0, 64 16.5 (17.7 before), 8 rows of x 16 to a block 21.0 and
// 64 19.1.
//
// More rows of x: a block takes more rows of w where there are enough of them
// to fill the chip all the same: x is then read by fewer blocks.  Of 28672 rows of
// 4096, 16 rows of x: 47 us with 64 rows in a block of 4 waves, 58 with 16 or 32.
//
// With a norm, which every block makes for itself, 16 rows of w share it: 768 to
// 2304, 1 row 3.6 us, 4.0 with 8 rows of w; deep rows, of which the loads are the
// longer part, 8: 4096 to 6144 13.0 and 14.3.
template <int MT, int ACT>
void pick(const SkinnyArgs& a, hipStream_t st) {
  constexpr bool PAIR = ACT == SKINNY_SWIGLU;
  const int tiles = (a.N + 15) / 16 * (PAIR ? 2 : 1);
  if constexpr (MT == 1) {
    const bool shallow = a.K < 2048 && tiles >= 1280;
    if (a.nw) {
      if (a.M <= 4 && (PAIR || a.K <= 2048)) launch_norm<4, ACT, 4>(a, st);
      else if (a.M <= 4) launch_norm<2, ACT, 4>(a, st);
      else if (a.M <= 8) launch_norm<2, ACT, 2>(a, st);
      else launch_norm<PAIR ? 2 : 1, ACT, 1>(a, st);
      return;
    }
    if constexpr (PAIR) {
      if (a.M <= 8) return launch<1, 2, 8, ACT, 0, 2>(a, st);
    } else {
      if (a.M <= 2 && shallow) return launch<1, 2, 8, ACT, 0, 4>(a, st);
      // rows of w up to which a block has four
      const int fours = a.M > 4 ? 0 : a.M > 2 ? 1024 : a.K < 2048 ? 2048
                        : a.M == 2 ? 6144 : a.N;
      if (a.N <= fours) return launch<1, 1, 8, ACT, 0, 4>(a, st);
      if (a.M <= 4 && a.N <= 2048) return launch<1, 2, 8, ACT, 0, 4>(a, st);
      if (a.M <= 8 && a.N <= 2048) return launch<1, 1, 8, ACT, 0, 2>(a, st);
      if (a.M <= 8 && !shallow) return launch<1, 2, 8, ACT, 0, 2>(a, st);
    }
  }
  if (tiles >= 1280) launch<MT, 4, 4, ACT>(a, st);
  else if (PAIR || (MT > 1 && tiles >= 384)) launch<MT, 2, 8, ACT>(a, st);
  else if constexpr (!PAIR) launch<MT, 1, 8, ACT>(a, st);
}

template <int ACT>
void pick(const SkinnyArgs& a, hipStream_t st) {
  if (a.M <= 16) pick<1, ACT>(a, st);
  else if (a.M <= 32) pick<2, ACT>(a, st);
  else pick<4, ACT>(a, st);
}

// The depth split over blocks too, for products whose N alone leaves a block
// to a compute unit only with few rows of w each, which then all read all of x.
// A block has 4 tiles of 16 rows of w, two waves to a tile, and one span of the
// depth; x comes through LDS, KC columns at a time, shared by all waves, the
// weights from memory to the wave that multiplies them, the next KC columns of
// both on their way meanwhile.  4096 rows of 4096 and of 14336 columns, in us,
// whole depths (or the library where that was faster) and split in 4: 16 rows
// of x 10.0 and 8.8, 26.2 and 23.5; 24 rows 12.8 and 9.6, 29.5 and 24.8; 64 rows
// 18.7 and 11.5, 39.2 and 30.0 (33 and 117 MB, read alone in 6.4 and 21.4); in 8,
// 64 rows 12.1 and 30.1, and the sums are read by 64 blocks of the next norm.
struct SplitArgs {
  SkinnyArgs s;
  float* sums;                   // [parts][M][N]
  int per;                       // columns of a span, a multiple of KC
};

template <int MT, int KC>
__global__ void __launch_bounds__(512)
skinny_split_kernel(SplitArgs g) {
  const SkinnyArgs& a = g.s;
  constexpr int T = 4, KS = 2, SPW = KC / 32 / KS;
  constexpr int ROWS = 16 * MT, LD = KC + 8;
  constexpr int XS = ROWS * KC / 8 / 512;
  static_assert(2 * ROWS * LD * 2 >= 8 * MT * 1024, "the sums share x's place");
  __shared__ __attribute__((aligned(16))) short lds[2 * ROWS * LD];
  const int tid = threadIdx.x, wid = tid >> 6, l = tid & 63;
  const int lr = l & 15, lg = l >> 4, t = wid % T, kg = wid / T;
  const int n0 = (blockIdx.x * T + t) * 16;
  const int k0 = blockIdx.y * g.per, k1 = min(a.K, k0 + g.per);
  const int chunks = (k1 - k0 + KC - 1) / KC;
  const short* wp = a.w + (long)min(n0 + lr, a.N - 1) * a.K;
  const int wc = k0 + kg * SPW * 32 + 8 * lg;

  f32x4 acc[MT];
  #pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Span { bf16x8 v[SPW]; };
  auto fetch_w = [&](Span& w, int c) {
    #pragma unroll
    for (int u = 0; u < SPW; ++u)
      w.v[u] = *(const bf16x8*)(wp + min(wc + c * KC + 32 * u, a.K - 8));
  };
  bf16x8 xr[XS];
  auto fetch_x = [&](int c) {
    #pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int s = i * 512 + tid, col = k0 + c * KC + s % (KC / 8) * 8;
      xr[i] = *(const bf16x8*)(a.x + min(s / (KC / 8), a.M - 1) * a.ldx +
                               min(col, a.K - 8));
    }
  };
  // columns behind the end count as zero on both sides
  auto put_x = [&](int c) {
    #pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int s = i * 512 + tid, col = k0 + c * KC + s % (KC / 8) * 8;
      *(bf16x8*)(lds + (c & 1) * ROWS * LD + s / (KC / 8) * LD + s % (KC / 8) * 8) =
          col < k1 ? xr[i] : bf16x8{};
    }
    // not __syncthreads(), which waits for the weights on their way too
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto use = [&](Span& w, int c) {
    if (k0 + (c + 1) * KC > k1) {
      #pragma unroll
      for (int u = 0; u < SPW; ++u)
        if (wc + c * KC + 32 * u >= k1) w.v[u] = bf16x8{};
    }
    const short* x = lds + (c & 1) * ROWS * LD + lr * LD + kg * SPW * 32 + 8 * lg;
    #pragma unroll
    for (int u = 0; u < SPW; ++u)
      #pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = mma(w.v[u], *(const bf16x8*)(x + m * 16 * LD + 32 * u), acc[m]);
  };
  Span w0, w1;
  fetch_x(0);
  fetch_w(w0, 0);
  put_x(0);
  for (int c = 0; c < chunks; c += 2) {
    if (c + 1 < chunks) {
      fetch_x(c + 1);
      fetch_w(w1, c + 1);
    }
    use(w0, c);
    if (c + 1 >= chunks) break;
    put_x(c + 1);
    if (c + 2 < chunks) {
      fetch_x(c + 2);
      fetch_w(w0, c + 2);
    }
    use(w1, c + 1);
    if (c + 2 < chunks) put_x(c + 2);
  }
  __syncthreads();
  f32x4(*part)[MT][64] = (f32x4(*)[MT][64])lds;      // [wave][m][lane]
  #pragma unroll
  for (int m = 0; m < MT; ++m) part[wid][m][l] = acc[m];
  __syncthreads();
  for (int m = kg; m < MT; m += KS) {
    f32x4 s = part[t][m][l] + part[T + t][m][l];
    const int row = 16 * m + lr, n = n0 + 4 * lg;
    if (row >= a.M || n >= a.N) continue;            // N is a multiple of 4
    if (a.bias && blockIdx.y == 0)
      #pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += bf2f(a.bias[n + j]);
    *(f32x4*)(g.sums + ((long)blockIdx.y * a.M + row) * a.N + n) = s;
  }
}

template <int MT, int KC>
void launch_split(const SkinnyArgs& a, float* sums, long parts, hipStream_t st) {
  SplitArgs g = {a, sums, (int)((a.K + parts * KC - 1) / (parts * KC) * KC)};
  const dim3 grid((a.N + 63) / 64, (unsigned)parts);
  hipLaunchKernelGGL((skinny_split_kernel<MT, KC>), grid, dim3(512), 0, st, g);
}

constexpr int split_chunk(int M) { return M <= 32 ? 512 : 256; }

}  // namespace

// Fewer than 16 MB of weights are read in the time of a launch or two, and up
// to 8 rows whole depths lose less than the reader pays for the sums (24.9 and
// 23.4 us of 14336 columns, 9.2 and 8.7 of 4096).  As many parts as give every
// compute unit a block.
long skinny_parts(const SkinnyArgs& a) {
  if (!skinny_takes(a) || a.nw || a.res || a.M <= 8 || a.N % 4 ||
      (long)a.N * a.K < 8l * 1024 * 1024)
    return 0;
  const long chunk = split_chunk(a.M), blocks = (a.N + 63) / 64;
  const long chunks = (a.K + chunk - 1) / chunk;
  const long want = std::min(std::max(1l, 256 / blocks), std::min(8l, chunks));
  const long per = (chunks + want - 1) / want;
  return (chunks + per - 1) / per;
}

// Where w has many rows, the blocks that take whole depths, or the library's tiles,
// fill the chip.  A step of two layers, whole (or the library) and split, in us:
// width 5120, feed-forward 13824, 17 rows 371 and 342, 64 rows 378 and 366; 6144 and
// 6144, 16 rows 315 and 292, 17 rows 279 and 286, 64 rows 318 and 327; 7168 and 8192,
// 16 rows 390 and 366; 8192 and 8192, 9 rows 381 and 404, 64 rows 404 and 432; 12288
// and 8192, 64 rows 683 and 786.  Depths of three times the rows of w and more are
// worth it a little longer: 6144 and 20480, 17 rows 641 and 528, 8192 and 28672, 48
// rows 937 and 834, but 7168 and 24576, 17 rows 582 and 616, 10240 and 32768, 33
// rows 1095 and 1211.
bool skinny_split_pays(const SkinnyArgs& a) {
  const bool deep = a.K >= 3l * a.N && a.N <= (a.M <= 32 ? 6144 : 8192);
  return a.N <= (a.M <= 16 ? 7168 : 5120) || deep;
}

void skinny_split(const SkinnyArgs& a, float* sums, long parts, hipStream_t st) {
  if (a.M <= 16) launch_split<1, split_chunk(16)>(a, sums, parts, st);
  else if (a.M <= 32) launch_split<2, split_chunk(32)>(a, sums, parts, st);
  else launch_split<4, split_chunk(64)>(a, sums, parts, st);
}

bool skinny_takes(const SkinnyArgs& a) {
  return a.M >= 1 && a.M <= 64 && a.N >= 1 && a.K >= 8 && a.K % 8 == 0 &&
         a.ldx % 8 == 0 && (size_t)a.x % 16 == 0 && (size_t)a.w % 16 == 0 &&
         (!a.nw || skinny_norms(a.M, a.K));
}

// A norm of few elements costs a block less than a launch of its own (2.8 us)
// would: in us, with the norm, and the product alone: 768 to 2304, 1 row 3.6 and 3.1, 10
// rows 4.2 and 3.4; 1024 to 4096, 8 rows 4.6 and 4.1; 4096 to 6144, 2 rows 13.1 and
// 11.5, 4 rows 13.6 and 12.9.  A wave holds up to four steps of the depth; with eight,
// 8 rows of 4096 to 6144 are 18.0 and 14.1, and behind much of the weights a launch is
// 4.9: as good.
bool skinny_norms(long M, long K) {
  return M >= 1 && K <= (M <= 4 ? 4096 : M <= 8 ? 2048 : M <= 16 ? 1024 : 0);
}

// Where the rows of w are many and deep, each of the several blocks of a compute
// unit norms again: 2048 to 2 x 5632, 1 row 11.6 and 9.8 without the norm, 4096 to 2 x
// 14336 48.4 and 41.0.  768 to 50257 takes 20.8 and 22.2, so the last norm of a model
// stays a launch.
bool skinny_norm_pays(long M, long K, SkinnyAct act) {
  return skinny_norms(M, K) && (act != SKINNY_SWIGLU || K <= 2048);
}

void skinny_gemm(SkinnyArgs a, SkinnyAct act, hipStream_t st) {
  auto fours = [&](const short* p, long ld) { return (size_t)p % 8 == 0 && ld % 4 == 0; };
  a.fours = a.N % 4 == 0 && fours(a.y, a.ldy) && fours(a.bias, 0) &&
            (!a.res || fours(a.res, a.ldr));
  if (act == SKINNY_GELU) pick<SKINNY_GELU>(a, st);
  else if (act == SKINNY_SWIGLU) pick<SKINNY_SWIGLU>(a, st);
  else pick<SKINNY_NONE>(a, st);
}

// x (M, K), w (N, K) or (2N, K) for act 2; act: 0 none, 1 gelu, 2 swiglu;
// norm_w, norm_b: of a norm of x before (no norm_b: RMS norm)
torch::Tensor skinny_linear(torch::Tensor x, torch::Tensor w,
                            c10::optional<torch::Tensor> bias,
                            c10::optional<torch::Tensor> res, long act,
                            c10::optional<torch::Tensor> norm_w,
                            c10::optional<torch::Tensor> norm_b, double eps) {
  CHECK_CUDA(x); CHECK_CUDA(w); CHECK_CONTIG(w);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) &&
              x.stride(1) == 1 && act >= 0 && act <= 2 &&
              (act != SKINNY_SWIGLU || w.size(0) % 2 == 0),
              "skinny_linear: shapes");
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16 &&
              w.scalar_type() == torch::kBFloat16, "skinny_linear: bf16 only");
  SkinnyArgs a = {};
  a.M = (int)x.size(0);
  a.N = (int)(w.size(0) / (act == SKINNY_SWIGLU ? 2 : 1));
  a.K = (int)x.size(1);
  auto y = torch::empty({a.M, a.N}, x.options());
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.y = (short*)y.data_ptr();
  a.ldx = x.stride(0);
  a.ldy = a.N;
  a.bias = a.res = nullptr;
  a.ldr = 0;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->is_contiguous() &&
                bias->numel() == a.N && act != SKINNY_SWIGLU &&
                bias->scalar_type() == torch::kBFloat16, "skinny_linear: bias");
    a.bias = (const short*)bias->data_ptr();
  }
  if (res.has_value()) {
    TORCH_CHECK(res->is_cuda() && res->dim() == 2 && res->stride(1) == 1 &&
                res->sizes() == y.sizes() &&
                res->scalar_type() == torch::kBFloat16, "skinny_linear: res");
    a.res = (const short*)res->data_ptr();
    a.ldr = res->stride(0);
  }
  if (norm_w.has_value()) {
    for (const auto* t : {&norm_w, &norm_b})
      TORCH_CHECK(!t->has_value() ||
                  ((*t)->is_cuda() && (*t)->is_contiguous() && (*t)->numel() == a.K &&
                   (size_t)(*t)->data_ptr() % 16 == 0 &&
                   (*t)->scalar_type() == torch::kBFloat16), "skinny_linear: norm");
    a.nw = (const short*)norm_w->data_ptr();
    a.nb = norm_b.has_value() ? (const short*)norm_b->data_ptr() : nullptr;
    a.eps = (float)eps;
  }
  TORCH_CHECK(skinny_takes(a), "skinny_linear: up to 64 aligned rows");
  skinny_gemm(a, (SkinnyAct)act, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return y;
}

// x (M, K), w (N, K), 9 to 64 rows and 16 MB of w or more: (parts, M, N) float32
torch::Tensor skinny_linear_parts(torch::Tensor x, torch::Tensor w,
                                  c10::optional<torch::Tensor> bias) {
  CHECK_CUDA(x); CHECK_CUDA(w); CHECK_CONTIG(w);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) &&
              x.stride(1) == 1 && x.scalar_type() == torch::kBFloat16 &&
              w.scalar_type() == torch::kBFloat16, "skinny_linear_parts: operands");
  TORCH_CHECK(!bias.has_value() ||
              (bias->is_cuda() && bias->is_contiguous() && bias->numel() == w.size(0) &&
               bias->scalar_type() == torch::kBFloat16), "skinny_linear_parts: bias");
  SkinnyArgs a = {};
  a.M = (int)x.size(0);
  a.N = (int)w.size(0);
  a.K = (int)x.size(1);
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.bias = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  a.ldx = x.stride(0);
  const long parts = skinny_parts(a);
  TORCH_CHECK(parts, "skinny_linear_parts: 9 to 64 rows, 16 MB of weights");
  auto sums = torch::empty({parts, a.M, a.N}, x.options().dtype(torch::kFloat32));
  skinny_split(a, sums.data_ptr<float>(), parts, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return sums;
}
