// y = x w^T for few rows x (a decode step: up to 64), bf16, float32 sums.
//
// What bounds it is reading w once.  A weight goes from memory to the one
// wave that multiplies it and nowhere else: a block has 16 rows of w (RT
// times that), its 8 waves split the depth in spans of 32 * U columns, and
// the rows of x, which every block reads, come out of the caches as the other
// operand of the 16x16x32 MFMA.  Each wave has the next span's loads in
// flight while it multiplies one.  The waves' sums meet in LDS at the end,
// where bias, residual, GELU or the gate's product join before the only
// rounding.

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
  return 0.5f * z * (2.f - 2.f / (__expf(2.f * u) + 1.f));
}

// Rows of x, normed (layer norm with a bias, else RMS norm) and rounded, into
// LDS; a wave takes a row at a time, up to 4096 columns.
template <int NW>
DEVINL void norm_rows(const SkinnyArgs& a, short* xs) {
  constexpr int NV = 8;
  const int wid = threadIdx.x >> 6, l = threadIdx.x & 63;
  const float inv = 1.f / (float)a.K;
  for (int m = wid; m < a.M; m += NW) {
    bf16x8 v[NV];
    float s = 0.f, mean = 0.f;
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = (n * 64 + l) * 8;
      if (n * 512 < a.K)
        v[n] = *(const bf16x8*)(a.x + m * a.ldx + min(c, a.K - 8));
    }
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const bool in = (n * 64 + l) * 8 < a.K;
      if (n * 512 < a.K)
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = in ? bf2f(v[n][j]) : 0.f;
          s += a.nb ? x : x * x;
        }
    }
    s = wave_reduce_sum(s) * inv;
    if (a.nb) {
      mean = s;
      s = 0.f;
      #pragma unroll
      for (int n = 0; n < NV; ++n) {
        const bool in = (n * 64 + l) * 8 < a.K;
        if (n * 512 < a.K)
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float d = in ? bf2f(v[n][j]) - mean : 0.f;
            s += d * d;
          }
      }
      s = wave_reduce_sum(s) * inv;
    }
    const float rstd = rsqrtf(s + a.eps);
    #pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = (n * 64 + l) * 8;
      if (c >= a.K) continue;
      const bf16x8 w = *(const bf16x8*)(a.nw + c);
      bf16x8 b = {}, o;
      if (a.nb) b = *(const bf16x8*)(a.nb + c);
      #pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = f2bf((bf2f(v[n][j]) - mean) * rstd * bf2f(w[j]) + bf2f(b[j]));
      *(bf16x8*)(xs + m * (a.K + 8) + c) = o;
    }
  }
}

// MT tiles of 16 rows of x, RT tiles of 16 rows of w (SWIGLU: half of them
// gate rows, half the up rows that go with them), NW waves.  NORM: the rows of
// x are normed first, by every block for itself, into LDS; the first weights
// are on their way meanwhile.
template <int MT, int RT, int NW, int ACT, bool NORM>
__global__ void __launch_bounds__(64 * NW)
skinny_kernel(SkinnyArgs a) {
  constexpr bool PAIR = ACT == SKINNY_SWIGLU;
  constexpr int U = MT + RT <= 3 ? 4 : 2;
  constexpr int SPAN = 32 * U;
  constexpr int OT = PAIR ? RT / 2 : RT;      // output tiles
  __shared__ __attribute__((aligned(16))) f32x4 part[NW][MT * RT][64];

  const int wid = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int lr = l & 15, lg = l >> 4;
  const int n0 = blockIdx.x * 16 * OT;
  const short *wp[RT], *xp[MT];
  #pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int n = min(n0 + 16 * (r % OT) + lr, a.N - 1) + (r / OT) * a.N;
    wp[r] = a.w + (long)n * a.K + 8 * lg;
  }
  extern __shared__ __attribute__((aligned(16))) short xs[];   // NORM: [M][K + 8]
  #pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = min(16 * m + lr, a.M - 1);
    xp[m] = (NORM ? xs + row * (a.K + 8) : a.x + (long)row * a.ldx) + 8 * lg;
  }

  f32x4 acc[MT][RT];
  #pragma unroll
  for (int m = 0; m < MT; ++m)
    #pragma unroll
    for (int r = 0; r < RT; ++r) acc[m][r] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Span { bf16x8 w[RT][U], x[NORM ? 1 : MT][U]; };
  auto fetch = [&](Span& s, int k0) {
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      #pragma unroll
      for (int r = 0; r < RT; ++r)
        s.w[r][u] = *(const bf16x8*)(wp[r] + k0 + 32 * u);
      if constexpr (!NORM)
        #pragma unroll
        for (int m = 0; m < MT; ++m) s.x[m][u] = *(const bf16x8*)(xp[m] + k0 + 32 * u);
    }
  };
  auto use = [&](const Span& s, int k0) {
    #pragma unroll
    for (int u = 0; u < U; ++u)
      #pragma unroll
      for (int m = 0; m < MT; ++m) {
        const bf16x8 x = NORM ? *(const bf16x8*)(xp[m] + k0 + 32 * u) : s.x[m][u];
        #pragma unroll
        for (int r = 0; r < RT; ++r) acc[m][r] = mma(s.w[r][u], x, acc[m][r]);
      }
  };
  const int full = a.K / SPAN;               // whole spans
  Span s0, s1;
  int i = wid;
  if (i < full) fetch(s0, i * SPAN);
  if constexpr (NORM) {
    norm_rows<NW>(a, xs);
    __syncthreads();
  }
  for (; i < full; i += 2 * NW) {
    if (i + NW < full) fetch(s1, (i + NW) * SPAN);
    use(s0, i * SPAN);
    if (i + NW >= full) break;
    if (i + 2 * NW < full) fetch(s0, (i + 2 * NW) * SPAN);
    use(s1, (i + NW) * SPAN);
  }
  // what is left of the depth, 32 columns at a time, by the waves that have
  // had one span less; columns behind the end are read at its last 8 and
  // count as zero on both sides
  const int left = (a.K - full * SPAN + 31) / 32;
  const int mine = (wid - full % NW + NW) % NW;
  if (mine < left) {
    const int k0 = full * SPAN + 32 * mine;
    const bool in = k0 + 8 * lg < a.K;
    const int c = in ? k0 : a.K - 8 - 8 * lg;
    bf16x8 wv[RT], xv[MT];
    #pragma unroll
    for (int r = 0; r < RT; ++r) wv[r] = *(const bf16x8*)(wp[r] + c);
    #pragma unroll
    for (int m = 0; m < MT; ++m) xv[m] = *(const bf16x8*)(xp[m] + c);
    #pragma unroll
    for (int r = 0; r < RT; ++r) wv[r] = in ? wv[r] : bf16x8{};
    #pragma unroll
    for (int m = 0; m < MT; ++m) {
      xv[m] = in ? xv[m] : bf16x8{};
      #pragma unroll
      for (int r = 0; r < RT; ++r) acc[m][r] = mma(wv[r], xv[m], acc[m][r]);
    }
  }
  #pragma unroll
  for (int m = 0; m < MT; ++m)
    #pragma unroll
    for (int r = 0; r < RT; ++r) part[wid][m * RT + r][l] = acc[m][r];
  __syncthreads();

  // a lane has 4 outputs in a row of one row of x
  for (int t = wid; t < MT * OT; t += NW) {
    const int m = t / OT, o = t % OT;
    f32x4 s = part[0][m * RT + o][l];
    #pragma unroll
    for (int v = 1; v < NW; ++v) s += part[v][m * RT + o][l];
    if constexpr (PAIR) {
      f32x4 up = part[0][m * RT + OT + o][l];
      #pragma unroll
      for (int v = 1; v < NW; ++v) up += part[v][m * RT + OT + o][l];
      #pragma unroll
      for (int j = 0; j < 4; ++j) s[j] = s[j] / (1.f + __expf(-s[j])) * up[j];
    }
    const int row = 16 * m + lr, n = n0 + 16 * o + 4 * lg;
    if (row >= a.M) continue;
    short* y = a.y + row * a.ldy + n;
    const short* res = a.res ? a.res + row * a.ldr + n : nullptr;
    bf16x4 out;
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = n + j < a.N;
      if (a.bias && in) s[j] += bf2f(a.bias[n + j]);
      if (ACT == SKINNY_GELU) s[j] = gelu_tanh(s[j]);
      if (res && in) s[j] += bf2f(res[j]);
      out[j] = f2bf(s[j]);
    }
    if (n + 4 <= a.N && a.ldy % 4 == 0 && (size_t)a.y % 8 == 0) {
      *(bf16x4*)y = out;
    } else {
      #pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < a.N) y[j] = out[j];
    }
  }
}

template <int MT, int RT, int NW, int ACT>
void launch(const SkinnyArgs& a, hipStream_t st) {
  constexpr int OT = ACT == SKINNY_SWIGLU ? RT / 2 : RT;
  const dim3 grid((a.N + 16 * OT - 1) / (16 * OT)), block(64 * NW);
  if constexpr (MT == 1) {
    if (a.nw) {
      hipLaunchKernelGGL((skinny_kernel<MT, RT, NW, ACT, true>), grid, block,
                         (size_t)a.M * (a.K + 8) * 2, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((skinny_kernel<MT, RT, NW, ACT, false>), grid, block, 0,
                     st, a);
}

// A block takes more rows of w where there are enough of them to fill the
// chip all the same: x is then read by fewer blocks.  Of 28672 rows of 4096,
// 16 rows of x: 49 us with 64 rows in a block of 4 waves, 58 with 16 or 32;
// 8 rows of x: 47 and 49 us.  Of 6144: 17 us with 16 rows a block, 16 with
// 32, 21 with 64; of 4096: 10 and 14 us.
template <int MT, int ACT>
void pick(const SkinnyArgs& a, hipStream_t st) {
  constexpr bool PAIR = ACT == SKINNY_SWIGLU;
  const int tiles = (a.N + 15) / 16 * (PAIR ? 2 : 1);
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

// A norm of few elements costs a block less than a launch of its own would:
// the first weights are on their way meanwhile, and a wave has one row or two.
// With the norm's launch, and without, in us: 768 to 2304, 1 row 5.8 and 4.8,
// 8 rows 6.5 and 5.1, 16 rows 6.7 and 6.9; 768 to 3072, 1 row 6.0 and 5.0;
// 4096 to 6144 and to 2 x 14336, 1 row 18.5 + 55.1 and 20.0 + 49.4, 2 rows
// 19.2 + 56.0 and 20.4 + 50.4.  Where the rows of w are many enough for
// several blocks a compute unit, each of them norms again: 768 to 50257 takes
// 20.8 and 22.2, so the last norm of a model stays a launch.
bool skinny_norms(long M, long K) {
  return M >= 1 && M <= 16 && K <= 4096 && M * K <= 8 * 1024;
}

void skinny_gemm(const SkinnyArgs& a, SkinnyAct act, hipStream_t st) {
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
