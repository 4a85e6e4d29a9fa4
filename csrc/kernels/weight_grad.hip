// dW[N][K] = sum over t of dY[t][N] X[t][K]: the weight gradient of a linear
// layer whose dW is small against the number of rows, so that tiles of dW
// alone leave most of the chip idle.
//
// The rows are split over as many parts as give a block to every compute unit;
// a part's sums stay float32 and are added in order by a second kernel.  A
// block has a tile of 256 x 256, its 8 waves 128 x 64 each.  Both operands lie
// with their rows along the sum, so they are staged as they are, by copies
// into LDS up to four stages ahead, and transposed by the reads, which are a
// stage ahead of the products: a wave that reads at a stage's barrier, as all
// then do, waits for most of what its products take.
//
// 16384 rows, library, this, this with its copies asked for at once and up to the last
// stage (behind which the compiler waits for all of them once a round), and with reads at
// the barrier too, in us: 3072 x 768 152, 85 (with the sums), 92 and 96, 2304 x 768 121, 66,
// 72 and 75, 768 x 768 92, 39, 40 and 42; 8192 rows, 4096 x 4096 235, 241 (1140 TF/s), 256 and
// 259.  Copies three stages ahead are 1 to 2 % slower.  The second kernel takes 11 of the
// first shape's, writing the parts, 66 MB, as much again.

#include "../common.h"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// A stage lies as units of 4 rows x 32 columns, 256 bytes: four lanes of a copy
// take 64 bytes of a row (with units of 16 columns, 32 bytes, 5 % slower, when
// stages were three ahead).  A transpose read takes 16 columns of a unit; odd quads of rows have
// its halves swapped, so that the two quads of half a wave's read lie in
// different banks.
constexpr int BT = 32;                  // rows of a stage
constexpr int NB = 5;                   // stages in LDS, all of it
constexpr int TILE = 256;               // of N and of K
constexpr int OPER = BT * TILE;         // elements of an operand's stage

struct WgradArgs {
  const short *dy, *x;
  float* part;                          // [parts][N][K]
  int T, N, K, per;                     // per: stages of a part
};

DEVINL f32x4_t mma(bf16x8 a, bf16x8 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, a),
      __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, b), c, 0, 0, 0);
}

__global__ void __launch_bounds__(512)
wgrad_kernel(WgradArgs a) {
  __shared__ __attribute__((aligned(16))) short s0[2 * OPER], s1[2 * OPER];
  __shared__ __attribute__((aligned(16))) short s2[2 * OPER], s3[2 * OPER];
  __shared__ __attribute__((aligned(16))) short s4[2 * OPER];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int wm = wid >> 2, wn = wid & 3, g = l >> 4, c = l & 15;

  // blocks of one part next to each other on one XCD: they share its rows
  const unsigned nwg = gridDim.x, q8 = nwg / 8, r8 = nwg % 8;
  const unsigned xcd = blockIdx.x % 8;
  const unsigned id = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) +
                      blockIdx.x / 8;
  const int gk = (a.K + TILE - 1) / TILE, gn = (a.N + TILE - 1) / TILE;
  const int part = id / (gn * gk), tile = id % (gn * gk);
  const int n0 = tile / gk * TILE, k0 = tile % gk * TILE;
  const int t0 = part * a.per * BT;
  const int t1 = min(a.T, t0 + a.per * BT);
  const int ns = (t1 - t0 + BT - 1) / BT;

  // a wave fills 2 x 4 units of either operand: slot s of 16 bytes
  unsigned pa[2], pb[2];
  #pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int s = (wid * 2 + i) * 64 + l;
    const int unit = s >> 4, quad = unit / (TILE / 32);
    const int row = quad * 4 + ((s >> 2) & 3);
    const int col = (unit % (TILE / 32)) * 32 + (((s >> 1) ^ quad) & 1) * 16 + (s & 1) * 8;
    pa[i] = 2u * ((unsigned)row * a.N + min(n0 + col, a.N - 8));
    pb[i] = 2u * ((unsigned)row * a.K + min(k0 + col, a.K - 8));
  }
  // rows behind the part's last read as zero, and stages behind it, so that what is on
  // its way is the same in every step: where it may be less, the compiler waits for all of
  // it once a round
  auto copy = [&](short* to, const short* from, int width, const unsigned* at, int s, int i) INLINE {
    const int row = min(t0 + s * BT, t1);
    const unsigned long base = (unsigned long)(from + (long)row * width);
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((unsigned long)same((unsigned)(base >> 32)) << 32 | same((unsigned)base)), 0,
        (int)same(2u * min(BT, t1 - row) * width), 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (__attribute__((address_space(3))) void*)(to + (wid * 2 + i) * 512), 16,
        at[i], 0, 0, 0);
  };
  auto image = [&](auto n) INLINE {
    constexpr int I = decltype(n)::value % NB;
    return I == 0 ? s0 : I == 1 ? s1 : I == 2 ? s2 : I == 3 ? s3 : s4;
  };
  // copy J of four of a stage
  auto part_of = [&](auto n, int s, auto j) INLINE {
    constexpr int J = decltype(j)::value;
    if constexpr (J < 2) copy(image(n), a.dy, a.N, pa, s, J);
    else copy(image(n) + OPER, a.x, a.K, pb, s, J - 2);
  };
  auto stage = [&](auto n, int s) INLINE {
    each<4>([&](auto j) INLINE { part_of(n, s, j); });
  };

  // this lane's quads are g and 4 + g: any order of a stage's rows will do.
  // Even sixteens of columns lie from e, odd ones from o.
  const int lane = g * (TILE / 16) * 64 + (c >> 2) * 32 + (c & 3) * 4;
  const int e = lane + (g & 1) * 16, o = lane + (1 - (g & 1)) * 16;
  f32x4_t acc[8][4] = {};
  bf16x4 fa[2][8][2], fb[2][4][2];        // of this stage and the next
  // read r of a stage's 24: eight for fb, then those for fa
  auto read = [&](auto odd, const short* img, auto n) INLINE {
    constexpr int X = decltype(odd)::value, R = decltype(n)::value;
    typedef __attribute__((address_space(3))) bf16x4* P;
    if constexpr (R < 8)
      fb[X][R / 2][R % 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (P)(img + OPER + wn * 256 + (R / 2 & 1 ? o : e) + R / 4 * 128 + R % 2 * 4096));
    else {
      constexpr int M = (R - 8) / 2;
      fa[X][M][R % 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (P)(img + wm * 512 + (M & 1 ? o : e) + M / 2 * 128 + R % 2 * 4096));
    }
  };
  // The copies of the stage after the next have arrived, in all waves, those of two
  // later ones may not; in a form that the compiler's own count takes notice of.
  auto turn = [&] INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f78);        // vmcnt(8)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto frag = [](const bf16x4 (&f)[2]) INLINE {
    return __builtin_shufflevector(f[0], f[1], 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // Stage s out of registers, while stage s + 1 is read from LDS, s + 2 and s + 3
  // are on their way and s + 4 is asked for, where s - 1 lay.
  auto step = [&](auto n, int s) INLINE {
    constexpr int I = decltype(n)::value, X = I & 1;
    const short* next = image(std::integral_constant<int, I + 1>{});
    each<8>([&](auto m) INLINE {
      constexpr int M = decltype(m)::value;
      each<3>([&](auto r) INLINE {
        read(std::integral_constant<int, !X>{}, next,
             std::integral_constant<int, 3 * M + decltype(r)::value>{});
      });
      const bf16x8 am = frag(fa[X][M]);
      each<4>([&](auto k) INLINE { acc[M][k] = mma(frag(fb[X][k]), am, acc[M][k]); });
      if constexpr (M % 2 == 0)
        part_of(std::integral_constant<int, I + 4>{}, s + 4, std::integral_constant<int, M / 2>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    turn();
  };
  using std::integral_constant;
  stage(integral_constant<int, 0>{}, 0);
  stage(integral_constant<int, 1>{}, 1);
  stage(integral_constant<int, 2>{}, 2);
  stage(integral_constant<int, 3>{}, 3);
  turn();
  each<24>([&](auto r) INLINE { read(integral_constant<int, 0>{}, s0, r); });
  static_assert(NB == 5, "ten steps a round");
  for (int s = 0;;) {
    step(integral_constant<int, 0>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 1>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 2>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 3>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 4>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 5>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 6>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 7>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 8>{}, s);
    if (++s == ns) break;
    step(integral_constant<int, 9>{}, s);
    if (++s == ns) break;
  }

  // a lane has four columns of a row
  float* to = a.part + (long)part * a.N * a.K;
  #pragma unroll
  for (int m = 0; m < 8; ++m)
    #pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int row = n0 + wm * 128 + m * 16 + c;
      const int col = k0 + wn * 64 + n * 16 + g * 4;
      if (row < a.N && col < a.K) *(f32x4_t*)(to + (long)row * a.K + col) = acc[m][n];
    }
}

__global__ void __launch_bounds__(256)
wgrad_sum_kernel(const float* __restrict__ part, short* __restrict__ dw,
                 long n8, int parts) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  f32x4_t s0 = {}, s1 = {};
  #pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const f32x4_t* v = (const f32x4_t*)(part + (p * n8 + i) * 8);
    s0 += v[0];
    s1 += v[1];
  }
  bf16x8 o;
  #pragma unroll
  for (int j = 0; j < 4; ++j) { o[j] = f2bf(s0[j]); o[4 + j] = f2bf(s1[j]); }
  *(bf16x8*)(dw + i * 8) = o;
}

}  // namespace

torch::Tensor weight_grad(torch::Tensor dy, torch::Tensor x) {
  CHECK_CUDA(dy); CHECK_CUDA(x); CHECK_CONTIG(dy); CHECK_CONTIG(x);
  TORCH_CHECK(dy.dim() == 2 && x.dim() == 2 && dy.size(0) == x.size(0) &&
              dy.scalar_type() == torch::kBFloat16 &&
              x.scalar_type() == torch::kBFloat16, "weight_grad: operands");
  WgradArgs a = {};
  const long T = x.size(0), N = dy.size(1), K = x.size(1);
  TORCH_CHECK(T >= 1 && N >= 8 && K >= 8 && N % 8 == 0 && K % 8 == 0 &&
              T < (1l << 30) && N < (1l << 24) && K < (1l << 24) &&
              (size_t)dy.data_ptr() % 16 == 0 && (size_t)x.data_ptr() % 16 == 0,
              "weight_grad: sizes");
  a.dy = (const short*)dy.data_ptr();
  a.x = (const short*)x.data_ptr();
  a.T = (int)T; a.N = (int)N; a.K = (int)K;
  const long tiles = ((N + TILE - 1) / TILE) * ((K + TILE - 1) / TILE);
  const long stages = (T + BT - 1) / BT;
  // a block per compute unit: more parts cost more than they fill
  long parts = std::min(std::max<long>(1, 256 / tiles), stages);
  a.per = (int)((stages + parts - 1) / parts);
  parts = (stages + a.per - 1) / a.per;
  auto dw = torch::empty({N, K}, x.options());
  auto part = torch::empty({parts, N, K}, x.options().dtype(torch::kFloat32));
  a.part = part.data_ptr<float>();
  auto st = scaffold_stream();
  hipLaunchKernelGGL(wgrad_kernel, dim3((unsigned)(tiles * parts)), dim3(512), 0, st, a);
  const long n8 = N * K / 8;
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0,
                     st, a.part, (short*)dw.data_ptr(), n8, (int)parts);
  HIP_CHECK(hipGetLastError());
  return dw;
}
