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
// In us, with bias, library and this: 100 rows of 768 to 3072, GELU behind it (two launches
// there) 10.3 and 6.5, 317 rows 11.9 and 6.8, 999 rows 19.1 and 10.5, 2536 rows 27.8 and 18.6;
// 768 to 2304, 317 rows 7.8 and 5.9, 999 11.5 and 9.4, 2536 15.7 and 15.1; 768 to 768, 999 rows
// 7.7 and 5.9, 2536 9.3 and 7.9; 3072 to 768, 999 rows 14.2 and 12.6, 2536 21.1 and 19.6; 2048
// to 8192, GELU behind it, 256 rows 27.4 and 16.4, 1024 rows 44.7 and 34.9; 2048 to 2048, 1500
// rows 19.2 and 16.5; 4096 to 6144, 256 rows 39.0 and 25.3.

#include "../common.h"
#include "tile_gemm.h"

namespace {

DEVINL f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  typedef __attribute__((ext_vector_type(8))) __bf16 v8;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

DEVINL float gelu_tanh(float z) {
  const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (2.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * u) + 1.f));
}

DEVINL float gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

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
  else if (tile == 2) launch<2, 4, 4, 2, 4, ACT>(a, st);
  else launch<4, 4, 2, 4, 3, ACT>(a, st);
}

// The tile, or -1 where a library is faster.  In us, library and this: little of all but the
// depth, 1024 from 4096, 256 rows 10.7 and 14.4, 400 13.8 and 14.6, 700 17.8 and 15.1; 768 to
// 768, 65 rows 4.8 and 5.4, 100 6.0 and 5.5.  Tiles of 128 x 128: 4096 from 4096, 700 rows 30.4
// and 31.6, 2048 from 8192, 1500 rows (192 tiles) 56 and 66, 1600 (208) 67.2 and 65.2, 1700
// 64 and 53, 2032 73 and 69, 4096 from 14336, 700 rows (192) 97 and 106, 850 (224) 131 and 121,
// 8192 from 4096, 500 rows (256) 43 and 40, 2048 from 2048 19.2 and 16.5.  Of 128 x 256
// with nothing behind them: 3072 from 1024, 1500 rows (144 tiles) 15.9 and 17.8, 2304 from 768,
// 2536 (180) 15.7 and 15.1; with a GELU, of which a launch is saved, 4096 from 1024, 1500 rows
// (192) 26.4 and 20.9, 3072 from 768, 4096 rows (384) 38.4 and 31.2, but 6400 from 1600, 1500
// rows (300) 44.5 and 49.4.
int tile_of(const TileArgs& a, TileAct act) {
  auto tiles = [&](long m, long n) { return (a.M + m - 1) / m * ((a.N + n - 1) / n); };
  const long few = tiles(64, 64);
  if (a.M < 96 || few * 32 < a.K) return -1;
  if (few <= 256) return 0;
  if (tiles(128, 64) <= 256) return 1;
  const long square = tiles(128, 128);
  if (square <= 256) return a.K <= 2048 || square >= 208 ? 2 : -1;
  const long wide = tiles(128, 256);
  if (act != TILE_NONE) return wide <= 256 || (wide <= 512 && a.K <= 1024) ? 3 : -1;
  return wide >= 180 && wide <= 256 && a.K <= 1024 ? 3 : -1;
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

// act(x w^T + b) of rows (..., K), act as TileAct; None: not what it is for
c10::optional<torch::Tensor> tile_linear(const torch::Tensor& x, const torch::Tensor& w,
                                         const c10::optional<torch::Tensor>& bias, long act) {
  // what a plain kernel would not see: gradients, transforms, tensors of Python classes,
  // modes that watch each call
  if (c10::impl::dispatch_mode_enabled()) return c10::nullopt;
  auto plain = [&](const torch::Tensor& t) {
    const auto keys = t.key_set();
    return t.is_cuda() && t.scalar_type() == torch::kBFloat16 && t.device() == x.device() &&
           !keys.has(c10::DispatchKey::Python) &&
           !keys.has(c10::DispatchKey::FuncTorchBatched) &&
           !keys.has(c10::DispatchKey::FuncTorchGradWrapper) &&
           t.layout() == c10::kStrided && !t._fw_grad(0).defined() &&
           !(at::GradMode::is_enabled() && t.requires_grad());
  };
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
  if (!tile_takes(a, (TileAct)act)) return c10::nullopt;
  auto shape = x.sizes().vec();
  shape.back() = a.N;
  auto y = torch::empty(shape, x.options());
  a.y = (short*)y.data_ptr();
  tile_gemm(a, (TileAct)act, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return y;
}
