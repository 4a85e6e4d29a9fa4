// y = act(x w^T + b) for rows of x in the hundreds, bf16, float32 sums: products whose
// tiles are about as many as the compute units, where a library has too few of them or
// splits the depth and adds up behind a second launch.
//
// What bounds it is not the matrix cores (up to half busy) but what a unit gets out of
// its XCD's cache, 90 KB a microsecond when all ask: 32 KB, the columns that a tile of 128 x
// 128 takes in a step, come in 0.38 us, their products take 0.21, the reads from LDS 0.12.
// So a block has the smallest tile with which all blocks run at once, copies go into LDS
// three stages ahead, as whole lines of 128 bytes, evenly spread between the products, and
// neighbouring tiles lie on one XCD: 8 down, then across.  Further than three stages ahead,
// by lines that a wave of its own asked for, and blocks that start at different columns are
// no faster; tiles of 256 x 256 are a third slower here than a library's.
//
// In us, with bias, library and this: 317 rows of 768 to 3072, GELU behind it (two launches
// there) 11.9 and 6.9, 999 rows 19.1 and 10.5, 2536 rows 28.5 and 21.0; 768 to 2304, 317 rows
// 7.9 and 5.9; 768 to 768, 777 rows 7.7 and 5.9, 2536 9.3 and 8.3; 3072 to 768, 777 rows 14.4 and
// 12.4, 2536 20.1 and 19.4; 2048 to 8192, GELU behind it, 256 rows 28.4 and 17.5, 1024 rows 46.0
// and 36.6; 2048 to 2048, 1600 rows 20.4 and 18.4; 4096 to 6144, 256 rows 37.4 and 24.7.

#include <c10/core/DeviceGuard.h>

#include "../common.h"
#include "../plain.h"
#include "tile_gemm.h"

namespace {

// MT x NT: 16 x 16 products of a wave; GM x GN waves; NB stages of 64 columns in LDS
template <int MT, int NT, int GM, int GN, int NB, int ACT>
__global__ void __launch_bounds__(64 * GM * GN)
tile_kernel(TileArgs a) {
  constexpr int WAVES = GM * GN, BM = 16 * MT * GM, BN = 16 * NT * GN, BK = 64;
  constexpr int XS = BM * BK, WS = BN * BK;          // elements of a stage
  constexpr int CX = BM / 8 / WAVES, CW = BN / 8 / WAVES, C = CX + CW;   // copies of a wave
  static_assert(CX * 8 * WAVES == BM && CW * 8 * WAVES == BN, "copies");
  static_assert(MT + NT <= MT * NT, "a read behind each product");
  static_assert(NB == 3 || NB == 4, "stages");
  __shared__ __attribute__((aligned(16))) short s0[XS + WS], s1[XS + WS];
  __shared__ __attribute__((aligned(16))) short s2[XS + WS], s3[NB > 3 ? XS + WS : 8];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int lr = l & 15, lg = l >> 4, wm = wid / GN, wn = wid % GN;

  // tiles of an XCD next to each other, 8 down, then across
  const unsigned nwg = gridDim.x, q8 = nwg / 8, r8 = nwg % 8, xcd = blockIdx.x % 8;
  const unsigned id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) +
                      blockIdx.x / 8;
  const unsigned gm = (a.M + BM - 1) / BM, gn = (a.N + BN - 1) / BN;
  const unsigned group = id / (8 * gn), high = min(8u, gm - 8 * group);
  const unsigned in = id - group * 8 * gn;
  const int m0 = (8 * group + in % high) * BM, n0 = in / high * BN;

  const int ns = a.K / BK;
  // copies: 8 rows of 8 chunks; chunk c of a row lies at c ^ f(row), so that the 16
  // rows of a read lie in different banks
  auto xplace = [](int row) INLINE { return row >> 1 & 7; };
  auto wplace = [](int row) INLINE { return (row >> 1 & 1) | (row >> 4 & 3) << 1; };
  unsigned xs[CX], ws[CW];
  #pragma unroll
  for (int i = 0; i < CX; ++i) {
    const int row = (i * WAVES + wid) * 8 + (l >> 3);
    xs[i] = 2 * ((unsigned)min(row, a.M - 1 - m0) * (unsigned)a.ldx +
                 8 * ((l & 7) ^ xplace(row)));
  }
  #pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int row = (i * WAVES + wid) * 8 + (l >> 3);
    ws[i] = 2 * ((unsigned)min(row, a.N - 1 - n0) * a.K +
                 8 * ((l & 7) ^ wplace(row)));
  }
  auto image = [&](auto n) INLINE {
    constexpr int I = decltype(n)::value % NB;
    return I == 0 ? s0 : I == 1 ? s1 : I == 2 ? s2 : s3;
  };
  // stages behind the last are read as zero, so that the loop has no tail
  auto copy = [&](short* to, const short* from, const unsigned* at, int s, int i) INLINE {
    const unsigned long u = (unsigned long)from;
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((unsigned long)same((unsigned)(u >> 32)) << 32 | same((unsigned)u)), 0,
        (int)same(s < ns ? 0xffffffffu : 0u),
        0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (__attribute__((address_space(3))) void*)(to + (i * WAVES + wid) * 512), 16,
        at[i], s * 2 * BK, 0, 0);
  };
  // copy j of stage s
  auto stage = [&](auto n, int s, auto j) INLINE {
    constexpr int J = decltype(j)::value;
    if constexpr (J < CX) copy(image(n), a.x + m0 * a.ldx, xs, s, J);
    else copy(image(n) + XS, a.w + (long)n0 * a.K, ws, s, J - CX);
  };

  // a lane's places: rows lr of x, rows 16 (lr / 4) + 4 t + lr % 4 of each 64 of w, so
  // that a lane has 16 outputs in a row
  static_assert(NT % 4 == 0, "64 rows of w");
  const int xr = wm * 16 * MT + lr, wr = wn * 16 * NT + 16 * (lr >> 2) + (lr & 3);
  const int xf = xplace(lr), wf = wplace(16 * (lr >> 2) + (lr & 3));
  f32x4 acc[MT][NT] = {};
  bf16x8 fx[2][MT], fw[2][NT];
  constexpr int READS = MT + NT;
  // read r of a half of a stage
  auto read = [&](auto half, const short* img, auto r) INLINE {
    constexpr int P = decltype(half)::value, R = decltype(r)::value;
    if constexpr (R < NT) {
      fw[P][R] = *(const bf16x8*)(img + XS + (wr + 64 * (R / 4) + 4 * (R % 4)) * BK +
                                  8 * ((4 * P + lg) ^ wf));
    } else if constexpr (R < READS) {
      constexpr int I = R - NT;
      fx[P][I] = *(const bf16x8*)(img + (xr + 16 * I) * BK + 8 * ((4 * P + lg) ^ xf));
    }
  };
  constexpr auto count = [](int vm) { return (vm & 15) | (vm >> 4) << 14 | 0x0070; };
  // everything read so far is here, and the next stage is, in all waves
  auto turn = [&] INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(count((NB - 2) * C));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> lo;
  constexpr integral_constant<int, 1> hi;
  // The copies of stage s + NB, which lies where s does, go out in the second half
  // of step s, as all waves have read s, and the first of step s + 1, evenly: a
  // unit takes 64 bytes a cycle, and a wave that asks for more waits.
  constexpr int Q = MT * NT, CA = (C + 1) / 2, CB = C - CA;
  auto step = [&](auto n, int s) INLINE {
    constexpr int I = decltype(n)::value;
    each<Q>([&](auto q) INLINE {
      constexpr int M = decltype(q)::value / NT, T = decltype(q)::value % NT;
      acc[M][T] = mma(fw[0][T], fx[0][M], acc[M][T]);
      read(hi, image(n), q);
      constexpr int J = decltype(q)::value * CB / Q;
      if constexpr (J != (decltype(q)::value + 1) * CB / Q)
        stage(integral_constant<int, I + NB - 1>{}, s - 1 + NB, integral_constant<int, CA + J>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    turn();
    each<Q>([&](auto q) INLINE {
      constexpr int M = decltype(q)::value / NT, T = decltype(q)::value % NT;
      acc[M][T] = mma(fw[1][T], fx[1][M], acc[M][T]);
      read(lo, image(integral_constant<int, I + 1>{}), q);
      constexpr int J = decltype(q)::value * CA / Q;
      if constexpr (J != (decltype(q)::value + 1) * CA / Q)
        stage(integral_constant<int, I + NB>{}, s + NB, integral_constant<int, J>{});
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  each<NB>([&](auto n) INLINE {
    constexpr int N = decltype(n)::value;
    each<N < NB - 1 ? C : CA>([&](auto j) INLINE { stage(n, N, j); });
  });
  // of what is on its way, the first stage has to be here
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(count((NB - 2) * C + CA));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  each<READS>([&](auto r) INLINE { read(lo, s0, r); });
  for (int s = 0; s < ns; s += NB)
    each<NB>([&](auto n) INLINE { step(n, s + n); });

  #pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + xr + 16 * i;
    if (m >= a.M) continue;
    #pragma unroll
    for (int g = 0; g < NT / 4; ++g) {
      const int n = n0 + wn * 16 * NT + 64 * g + 16 * lg;
      #pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (n + 8 * h >= a.N) continue;            // N is a multiple of 8
        bf16x8 b = {};
        if (a.bias) b = *(const bf16x8*)(a.bias + n + 8 * h);
        float y[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          y[j] = acc[i][4 * g + 2 * h + j / 4][j % 4] + bf2f(b[j]);
          if (ACT == TILE_GELU_TANH) y[j] = gelu_tanh(y[j]);
          if (ACT == TILE_GELU_ERF) y[j] = gelu_erf(y[j]);
        }
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        *(u32x4*)(a.y + (long)m * a.ldy + n + 8 * h) =
            u32x4{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3]),
                  cvt_pk_bf16(y[4], y[5]), cvt_pk_bf16(y[6], y[7])};
      }
    }
  }
}

template <int MT, int NT, int GM, int GN, int NB, int ACT>
void launch(const TileArgs& a, hipStream_t st) {
  constexpr int BM = 16 * MT * GM, BN = 16 * NT * GN;
  const long tiles = (long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((tile_kernel<MT, NT, GM, GN, NB, ACT>), dim3((unsigned)tiles),
                     dim3(64 * GM * GN), 0, st, a);
}

template <int ACT>
void pick(const TileArgs& a, int tile, hipStream_t st) {
  if (tile == 0) launch<2, 4, 2, 1, 4, ACT>(a, st);
  else if (tile == 1) launch<2, 4, 4, 1, 4, ACT>(a, st);
  else if (ACT == TILE_NONE || tile == 2) launch<2, 4, 4, 2, 4, ACT>(a, st);
  else if constexpr (ACT != TILE_NONE) launch<4, 4, 2, 4, 3, ACT>(a, st);
}

// The tile, or -1 where a library is faster: the lines lie where of 3000 sizes of 96 to 8192
// rows, N and K up to 28672 and 14336, next to none is slower.  In us, library and this, with
// a bias.
//
// A product alone.  Few tiles of some depth, which a library splits: 768 to 768, 160 rows (36 tiles
// of 64 x 64) 4.9 and 5.5, 777 rows (156) 7.7 and 5.9; 1024 from 8192, 1200 rows 43.0 and 49.1;
// 2048 from 5632, 640 rows 31.1 and 36.5; 768 from 3072, 2536 rows (240 of 128 x 64) 20.1 and 19.4;
// 6144 from 4096, 256 rows 37.4 and 24.7.  Depths that leave much of a round of four stages:
// 1280 from 576, 140 rows 4.7 and 5.4, 3328 from 64, 272 rows 4.1 and 5.0.  Rows that leave much of
// a tile's 128: 7104 from 2944, 142 rows 18.0 and 19.6.  Tiles of 128 x 128: 2048 from 2048, 1600
// rows (208) 20.4 and 18.4, but 4096 from 1024, 900 rows (256) 13.7 and 15.4, 1152 from 4736, 3437
// rows (243) 39.7 and 41.4.  128 x 256: 2304 from 768, 2536 rows (180) 16.2 and 15.5, 3072 from
// 768, 2536 rows (240) 17.7 and 19.4.  Without a bias tiles of 128 x 128 end sooner: 2048 from
// 2048, 2032 rows (256) 20.8 and 19.6, with one 22.2 and 22.8; and deep ones that fill the chip
// and are no strip, 250 to 256 tiles, are faster: of 78 sizes of 2304 to 8192 the mean is 0.95 of
// the library's, strips of 3 to 7 tiles up to 1.11 of it, others 1.02; 2048 from 8192, 2032 rows,
// 68.7 and 67.3, between the kernels of a model 73.4 and 62.9.
//
// With a GELU behind it a launch and a pass over memory are saved: 768 to 3072, 2536 rows (240
// of 128 x 256) 28.5 and 21.0, 4096 rows (384) 39.3 and 33.2; 8192 from 2048, 1024 rows (256) 46.0
// and 36.6; 6144 from 4096, 256 rows 41.1 and 25.5; but 1600 from 6400, 640 rows 31.1 and 32.0,
// 2536 rows 75 and 85; 4096 from 14336, 1400 rows 176 and 193; 1664 from 704, 4843 rows (266)
// 27.2 and 28.9.
int tile_of(const TileArgs& a, TileAct act) {
  auto tiles = [&](long m, long n) { return (a.M + m - 1) / m * ((a.N + n - 1) / n); };
  const long few = tiles(64, 64), tall = tiles(128, 64), square = tiles(128, 128);
  const int K = a.K, stages = K / 64;
  if (a.M < 96) return -1;
  if (act != TILE_NONE) {
    if (few <= 256) return few * 32 >= K && K <= 6144 ? 0 : -1;
    if (tall <= 256) return K <= 4096 || (tall >= 208 && K <= 8192) ? 1 : -1;
    if (square <= 256) return K <= 2048 || (square >= 208 && K <= 8192) ? 2 : -1;
    const long wide = tiles(128, 256);
    if (wide <= 256)
      return K <= 1024 || (wide >= (K <= 2048 ? 160 : 192) && K <= 8192) ? 3 : -1;
    return wide <= 512 && K <= (wide >= 384 ? 768 : 576) ? 3 : -1;
  }
  if ((stages + 3) / 4 * 4 * 7 > stages * 8) return -1;
  if (few <= 256) return few >= (K <= 512 ? 1 : 32 + K / 32) && K <= 5120 ? 0 : -1;
  if ((a.M + 127) / 128 * 128l * 3 > a.M * 4l) return -1;
  if (tall <= 256) return K <= 2048 || (tall >= 192 && K <= 4096) ? 1 : -1;
  if (K > 2048)
    return !a.bias && K <= 8192 && square >= 250 && square <= 256 && a.M > 7 * 128 &&
                   a.N > 7 * 128 ? 2 : -1;
  return square <= (a.bias ? 223 : K <= 1024 ? 239 : 256) && (K <= 1024 || square >= 160)
             ? 2 : -1;
}

}  // namespace

bool tile_takes(const TileArgs& a, TileAct act) {
  return a.M >= 1 && a.N >= 8 && a.N % 8 == 0 && a.K >= 64 && a.K % 64 == 0 &&
         a.K <= 1 << 22 && a.ldx % 8 == 0 && a.ldx >= a.K && a.ldx <= 1 << 22 &&
         a.ldy % 8 == 0 && ((size_t)a.x | (size_t)a.w | (size_t)a.y | (size_t)a.bias) % 16 == 0 &&
         tile_of(a, act) >= 0;
}

void tile_gemm(const TileArgs& a, TileAct act, hipStream_t st) {
  const int tile = tile_of(a, act);
  if (act == TILE_GELU_TANH) pick<TILE_GELU_TANH>(a, tile, st);
  else if (act == TILE_GELU_ERF) pick<TILE_GELU_ERF>(a, tile, st);
  else pick<TILE_NONE>(a, tile, st);
}

// Whether an autograd function in torch's place is worth it for x w^T + res, through which
// gradients go.  Where the product is a kernel's of ours the host takes no longer: both ways,
// eager, 134 us of torch's and 126 at 666 x 3072 x 768, 123 at 3125.  Where only a gradient is, it
// takes 13 to 30 us more, which the GPU has to have saved.  The large products' kernel: of 24
// sizes of more than 20 G products every one is faster (885 x 4096 x 8192 194 and 172 us); of 22 of
// 10 to 20 the mean is 0.93 and eight are 2 to 11 % slower (777 x 4096 x 4096 110 and 102, 890 x 2048
// x 8192 130 and 143, whose GPU time is 118 and 107); of less they are 6 to 11 % slower (408 x 2048
// x 5632 128 and 142, of the GPU 84 and 68).  Weight gradients of few tiles, for which a library's
// time grows with the rows: 43764 x 344 x 712 347 and 202, 22184 x 456 x 480 202 and 159, 51357 x 64
// x 96 180 and 162, of 29 sizes 0.71; of 43 below the line 1.03 (10381 x 488 x 432 147 and 164,
// 25997 x 576 x 80 154 and 164).
bool residual_takes(const torch::Tensor& x, const torch::Tensor& w, const torch::Tensor& res) {
  if (watched() || !x.is_cuda() || !memory(x, x.device()) || !memory(w, x.device()) ||
      !memory(res, x.device()) || x.dim() < 1 || w.dim() != 2 || res.dim() != x.dim())
    return false;
  const long N = w.size(0), K = w.size(1);
  if (N < 1 || N >= 1 << 30 || K < 1 || K > 1 << 22 || x.size(-1) != K || res.size(-1) != N)
    return false;
  const long M = x.numel() / K;
  if (M < 1 || M >= 1 << 30 ||
      res.sizes().slice(0, res.dim() - 1) != x.sizes().slice(0, x.dim() - 1))
    return false;
  TileArgs a = {};
  a.M = (int)M; a.N = (int)N; a.K = (int)K;
  a.ldx = K; a.ldy = N;
  if ((K <= BIG_DEPTH_OF_TRAINING && big_takes(a, TILE_NONE)) || tile_takes(a, TILE_NONE))
    return true;
  const bool dx = x.requires_grad(), dw = w.requires_grad();
  if ((double)M * (double)N * (double)K >= 10e9 &&
      ((dx && input_grad_takes(M, N, K)) || (dw && weight_grad_takes(M, N, K))))
    return true;
  // weight_grad.hip's
  const long small = std::min(N, K), large = std::max(N, K);
  return dw && (M >= 32768 || (M >= 8192 && M * (N + K) >= 20000000)) && N % 8 == 0 &&
         K % 8 == 0 && small >= 64 && (small >= 256 || large <= 8192) &&
         ((N + 255) / 256) * ((K + 255) / 256) <= 64;
}

// act(x w^T + b) of rows (..., K), act as TileAct, by these or by large tiles; None: not
// what they are for
c10::optional<torch::Tensor> tile_linear(const torch::Tensor& x, const torch::Tensor& w,
                                         const c10::optional<torch::Tensor>& bias, long act,
                                         bool grad) {
  // what a plain kernel would not see: gradients, transforms, tensors of Python classes
  if (watched()) return c10::nullopt;
  auto plain = [&](const torch::Tensor& t) { return ::plain(t, x.device()); };
  if (!x.defined() || x.dim() < 2 || w.dim() != 2 || act < 0 || act > 2 || !plain(x) || !plain(w) ||
      (bias.has_value() && !plain(*bias)) || x.size(-1) != w.size(1) || !w.is_contiguous() ||
      x.stride(-1) != 1 || (x.dim() > 2 && !x.is_contiguous()) ||
      (bias.has_value() &&
       (bias->dim() != 1 || !bias->is_contiguous() || bias->size(0) != w.size(0))) ||
      x.numel() == 0 || w.size(0) >= 1 << 30 || x.numel() / w.size(1) >= 1 << 30)
    return c10::nullopt;
  TileArgs a = {};
  a.K = (int)w.size(1);
  a.N = (int)w.size(0);
  a.M = (int)(x.numel() / a.K);
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.bias = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  a.ldx = x.dim() == 2 ? x.stride(0) : a.K;
  a.ldy = a.N;
  const bool big = (!grad || a.K <= BIG_DEPTH_OF_TRAINING) && big_takes(a, (TileAct)act) &&
                   (act != TILE_NONE || big_alone(a));
  if (!big && !tile_takes(a, (TileAct)act)) return c10::nullopt;
  // the operands' device, whichever is current: torch's product goes by it too
  const c10::DeviceGuard guard(x.device());
  auto shape = x.sizes().vec();
  shape.back() = a.N;
  auto y = torch::empty(shape, x.options());
  a.y = (short*)y.data_ptr();
  if (big) big_gemm(a, (TileAct)act, scaffold_stream());
  else tile_gemm(a, (TileAct)act, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return y;
}
