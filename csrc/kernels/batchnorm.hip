// Fused bf16 NHWC BatchNorm (+ReLU, +residual) for the ResNet headline
// config.  Without them the step spent 38% in MIOpen's fp32 BatchNorm
// kernels and 19% more in the bf16<->fp32 cast copies its fp32-only
// interface forces, vs ~30% in the convs themselves
// (profiles/resnet_kstats_r2.txt).  These kernels read/write the bf16 activation
// DIRECTLY (fp32 arithmetic inside), and fold the adjacent elementwise
// ops into the same pass:
//   fwd:  y = relu?(gamma*xhat + beta [+ res])     xhat=(x-mean)*rstd
//   bwd:  dy_eff = dy * (pre-relu > 0); dbeta = sum(dy_eff);
//         dgamma = sum(dy_eff*xhat);
//         dx = gamma*rstd*(dy_eff - dbeta/R - xhat*dgamma/R); dres = dy_eff
//         (the mask is recomputed from x, or, behind a residual, kept as one
//         bit per element, so that the residual is neither saved nor read)
//
// What bounds these is memory: 256 x 256 x 56 x 56 with a residual is 10.1
// passes over 411 MB, 657 us.  A thread has UN rows' loads in flight at a time, and
// every second pass walks the rows backwards, so that it starts with what
// the pass before has left in the memory-side cache.  Few rows are bound by
// launches instead: there one launch per direction does everything
// (bn_small_*).
//
// Layout: channels_last (N,C,H,W) = physical [R][C] bf16 with C
// contiguous, R = N*H*W; per-channel params/stats fp32.  Stats and
// backward reductions are two-stage column reduces (the colsum
// pattern) with bf16x8-vectorized row traffic (G13).

#include "../common.h"

namespace {

typedef short bf16x8_t __attribute__((ext_vector_type(8)));

struct F8 { float v[8]; };

DEVINL F8 up8(bf16x8_t x) {
  F8 r;
  #pragma unroll
  for (int j = 0; j < 8; ++j) r.v[j] = bf2f(x[j]);
  return r;
}

// thread -> (vector-column, row-group) map: CV = C/8 vector columns.
// CV <= 256: one block in x, G = 256/CV row-threads per column.
// CV > 256: gridDim.x column blocks, G = 1.
struct ColMap {
  int vc;     // global vector column (-1 = idle)
  int g;      // row-group index within block
  int G;      // row-groups per block
};

DEVINL ColMap colmap(int C) {
  const int CV = C / 8;
  ColMap m;
  if (CV >= 256) {
    m.vc = blockIdx.x * 256 + (int)threadIdx.x;
    m.g = 0;
    m.G = 1;
    if (m.vc >= CV) m.vc = -1;
  } else {
    m.G = 256 / CV;
    m.vc = (int)threadIdx.x % CV;
    m.g = (int)threadIdx.x / CV;
    // tail threads when CV does not divide 256 would re-walk other
    // groups' rows — idle them (all ResNet C are powers of two, but
    // the kernel must not silently double-count for other C)
    if (m.g >= m.G) m.vc = -1;
  }
  return m;
}

// Rows r0, r0 + step, ... below end of a pass, UN at a time: load(u, row) for all of
// them first, then use(u, row).  Backwards: from the last of R rows to the first.
template <int UN, bool BACK, typename L, typename U>
DEVINL void walk(long r0, long step, long end, long R, L load, U use) {
  auto row = [&](long r) { return BACK ? R - 1 - r : r; };
  long r = r0;
  for (; r + (UN - 1) * step < end; r += UN * step) {
    #pragma unroll
    for (int u = 0; u < UN; ++u) load(u, row(r + u * step));
    #pragma unroll
    for (int u = 0; u < UN; ++u) use(u, row(r + u * step));
  }
  for (; r < end; r += step) {
    load(0, row(r));
    use(0, row(r));
  }
}

// Sums of a block's row-groups, in a fixed order (float atomics would vary
// from run to run): out[0][C], out[1][C].
DEVINL void fold(const ColMap& m, int C, const float (&s)[8],
                 const float (&q)[8], float (&acc)[2][2048], float* out) {
  if (m.G == 1) {
    if (m.vc >= 0)
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        out[m.vc * 8 + j] = s[j];
        out[C + m.vc * 8 + j] = q[j];
      }
    return;
  }
  if (m.vc >= 0) {
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[0][m.g * C + m.vc * 8 + j] = s[j];
      acc[1][m.g * C + m.vc * 8 + j] = q[j];
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * C; i += 256) {
    const float* a = i < C ? acc[0] : acc[1];
    const int c = i < C ? i : i - C;
    float t = 0.f;
    for (int g = 0; g < m.G; ++g) t += a[g * C + c];
    out[i] = t;
  }
}

// ---- fwd stats: partial sum / sumsq per channel -> mid[ns][2][C]
template <int UN>
__global__ void __launch_bounds__(256)
bn_stats_kernel(const short* __restrict__ x, float* __restrict__ mid,
                long R, int C) {
  __shared__ float acc[2][2048];
  const ColMap m = colmap(C);
  float s[8] = {}, q[8] = {};
  if (m.vc >= 0) {
    bf16x8_t xs[UN];
    walk<UN, false>((long)blockIdx.y * m.G + m.g, (long)gridDim.y * m.G, R, R,
        [&](int u, long r) { xs[u] = *(const bf16x8_t*)(x + r * C + m.vc * 8); },
        [&](int u, long) {
          const F8 xv = up8(xs[u]);
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            s[j] += xv.v[j];
            q[j] += xv.v[j] * xv.v[j];
          }
        });
  }
  fold(m, C, s, q, acc, mid + ((long)blockIdx.y * 2) * C);
}

// Both sums of 16 channels over the slices, by 16 groups of lanes with 8
// slices' loads in flight.
DEVINL void final_sums(const float* __restrict__ mid, int ns, int C,
                       float (&acc)[2][16][16], float& s, float& q) {
  const int cl = (int)threadIdx.x & 15, g = (int)threadIdx.x >> 4;
  const int c = blockIdx.x * 16 + cl;
  s = q = 0.f;
  if (c < C) {
    #pragma unroll 8
    for (int i = g; i < ns; i += 16) {
      s += mid[((long)i * 2) * C + c];
      q += mid[((long)i * 2 + 1) * C + c];
    }
  }
  acc[0][g][cl] = s;
  acc[1][g][cl] = q;
  __syncthreads();
  s = q = 0.f;
  #pragma unroll
  for (int j = 0; j < 16; ++j) {
    s += acc[0][j][cl];
    q += acc[1][j][cl];
  }
}

struct StatsOut {
  float *mean, *rstd, *rmean, *rvar;
  float momentum, eps;
};

// mean, 1/std and the running statistics of a channel
DEVINL void put_stats(const StatsOut& o, int c, float mu, float var, long R) {
  var = fmaxf(var, 0.f);
  o.mean[c] = mu;
  o.rstd[c] = rsqrtf(var + o.eps);
  if (o.rmean) {
    // torch semantics: running update uses the UNBIASED batch variance
    const float ub = (R > 1) ? var * (float)R / (float)(R - 1) : var;
    o.rmean[c] = (1.f - o.momentum) * o.rmean[c] + o.momentum * mu;
    o.rvar[c] = (1.f - o.momentum) * o.rvar[c] + o.momentum * ub;
  }
}

__global__ void __launch_bounds__(256)
bn_stats_final_kernel(const float* __restrict__ mid, StatsOut o, int ns,
                      long R, int C) {
  __shared__ float acc[2][16][16];
  float s, q;
  final_sums(mid, ns, C, acc, s, q);
  const int c = blockIdx.x * 16 + ((int)threadIdx.x & 15);
  if (threadIdx.x >= 16 || c >= C) return;
  const float mu = s / (float)R;
  put_stats(o, c, mu, q / (float)R - mu * mu, R);
}

// ---- apply: y = relu?(gamma*xhat + beta [+ res]), and the sign's bit
struct Channel8 {
  float mu[8], rs[8], ga[8], be[8];
  DEVINL Channel8(int vc, const float* mean, const float* rstd, const float* w,
                  const float* b) {
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      mu[j] = mean[vc * 8 + j];
      rs[j] = rstd[vc * 8 + j];
      ga[j] = w[vc * 8 + j];
      be[j] = b[vc * 8 + j];
    }
  }
};

template <bool RELU, bool RES>
DEVINL bf16x8_t bn_out(const Channel8& p, bf16x8_t x, bf16x8_t res,
                       unsigned& bits) {
  const F8 xv = up8(x);
  bf16x8_t out;
  bits = 0;
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    float v = p.ga[j] * ((xv.v[j] - p.mu[j]) * p.rs[j]) + p.be[j];
    if (RES) v += bf2f(res[j]);
    if (RELU) {
      bits |= (v > 0.f ? 1u : 0u) << j;
      v = fmaxf(v, 0.f);
    }
    out[j] = f2bf(v);
  }
  return out;
}

// PAST: see past_caches()
template <bool RELU, bool RES, bool PAST>
__global__ void __launch_bounds__(256)
bn_apply_kernel(const short* __restrict__ x, const short* __restrict__ res,
                const float* __restrict__ mean, const float* __restrict__ rstd,
                const float* __restrict__ w, const float* __restrict__ b,
                short* __restrict__ y, unsigned char* __restrict__ mask,
                long R, int C, long span) {
  constexpr int UN = 2;
  const ColMap m = colmap(C);
  if (m.vc < 0) return;
  const Channel8 p(m.vc, mean, rstd, w, b);
  bf16x8_t xs[UN], rs[UN];
  const long r0 = (long)blockIdx.y * span;
  walk<UN, true>(r0 + m.g, m.G, min(R, r0 + span), R,
      [&](int u, long r) {
        xs[u] = *(const bf16x8_t*)(x + r * C + m.vc * 8);
        if (RES) rs[u] = get_from<PAST>((const bf16x8_t*)(res + r * C + m.vc * 8));
      },
      [&](int u, long r) {
        unsigned bits;
        put_to<PAST>((bf16x8_t*)(y + r * C + m.vc * 8), bn_out<RELU, RES>(p, xs[u], rs[u], bits));
        if (RELU && RES) mask[r * (C / 8) + m.vc] = (unsigned char)bits;
      });
}

// xhat and what of dy passes the ReLU.  MASK: its bits are kept, else the
// sign is that of gamma*xhat + beta.
template <bool RELU, bool MASK>
DEVINL void bn_grad(const Channel8& p, bf16x8_t dy, bf16x8_t x, unsigned bits,
                    float (&d)[8], float (&xh)[8]) {
  const F8 dv = up8(dy), xv = up8(x);
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    xh[j] = (xv.v[j] - p.mu[j]) * p.rs[j];
    d[j] = dv.v[j];
    if (MASK) d[j] = bits >> j & 1 ? d[j] : 0.f;
    else if (RELU) d[j] = p.ga[j] * xh[j] + p.be[j] > 0.f ? d[j] : 0.f;
  }
}

// ---- bwd reduce: partial sum(dy_eff), sum(dy_eff * xhat) -> mid
template <bool RELU, bool MASK>
__global__ void __launch_bounds__(256)
bn_bwd_reduce_kernel(const short* __restrict__ dy, const short* __restrict__ x,
                     const unsigned char* __restrict__ mask,
                     const float* __restrict__ mean,
                     const float* __restrict__ rstd,
                     const float* __restrict__ w, const float* __restrict__ b,
                     float* __restrict__ mid, long R, int C) {
  constexpr int UN = 4;
  __shared__ float acc[2][2048];
  const ColMap m = colmap(C);
  float sd[8] = {}, sx[8] = {};
  if (m.vc >= 0) {
    const Channel8 p(m.vc, mean, rstd, w, b);
    bf16x8_t ds[UN], xs[UN];
    unsigned ms[UN];
    walk<UN, false>((long)blockIdx.y * m.G + m.g, (long)gridDim.y * m.G, R, R,
        [&](int u, long r) {
          ds[u] = *(const bf16x8_t*)(dy + r * C + m.vc * 8);
          xs[u] = *(const bf16x8_t*)(x + r * C + m.vc * 8);
          if (MASK) ms[u] = mask[r * (C / 8) + m.vc];
        },
        [&](int u, long) {
          float d[8], xh[8];
          bn_grad<RELU, MASK>(p, ds[u], xs[u], ms[u], d, xh);
          #pragma unroll
          for (int j = 0; j < 8; ++j) {
            sd[j] += d[j];
            sx[j] += d[j] * xh[j];
          }
        });
  }
  fold(m, C, sd, sx, acc, mid + ((long)blockIdx.y * 2) * C);
}

__global__ void __launch_bounds__(256)
bn_bwd_final_kernel(const float* __restrict__ mid, float* __restrict__ dw,
                    float* __restrict__ db, int ns, int C) {
  __shared__ float acc[2][16][16];
  float sd, sx;
  final_sums(mid, ns, C, acc, sd, sx);
  const int c = blockIdx.x * 16 + ((int)threadIdx.x & 15);
  if (threadIdx.x >= 16 || c >= C) return;
  db[c] = sd;
  dw[c] = sx;
}

// ---- bwd dx (+ dres): dx = gamma*rstd*(dy_eff - db/R - xhat*dw/R)
template <bool RELU, bool MASK>
DEVINL bf16x8_t bn_dx(const Channel8& p, const float (&mdb)[8],
                      const float (&mdw)[8], bf16x8_t dy, bf16x8_t x,
                      unsigned bits, bf16x8_t& dres) {
  float d[8], xh[8];
  bn_grad<RELU, MASK>(p, dy, x, bits, d, xh);
  bf16x8_t dx;
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    dres[j] = d[j] == 0.f ? (short)0 : dy[j];
    dx[j] = f2bf(p.ga[j] * p.rs[j] * (d[j] - mdb[j] - xh[j] * mdw[j]));
  }
  return dx;
}

template <bool RELU, bool MASK, bool PAST>
__global__ void __launch_bounds__(256)
bn_bwd_dx_kernel(const short* __restrict__ dy, const short* __restrict__ x,
                 const unsigned char* __restrict__ mask,
                 const float* __restrict__ mean,
                 const float* __restrict__ rstd, const float* __restrict__ w,
                 const float* __restrict__ b, const float* __restrict__ dw,
                 const float* __restrict__ db, short* __restrict__ dx,
                 short* __restrict__ dres, long R, int C, long span) {
  constexpr int UN = 2;
  const ColMap m = colmap(C);
  if (m.vc < 0) return;
  const float invR = 1.f / (float)R;
  const Channel8 p(m.vc, mean, rstd, w, b);
  float mdb[8], mdw[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    mdb[j] = db[m.vc * 8 + j] * invR;
    mdw[j] = dw[m.vc * 8 + j] * invR;
  }
  bf16x8_t ds[UN], xs[UN];
  unsigned ms[UN];
  const long r0 = (long)blockIdx.y * span;
  walk<UN, true>(r0 + m.g, m.G, min(R, r0 + span), R,
      [&](int u, long r) {
        ds[u] = *(const bf16x8_t*)(dy + r * C + m.vc * 8);
        xs[u] = *(const bf16x8_t*)(x + r * C + m.vc * 8);
        if (MASK) ms[u] = mask[r * (C / 8) + m.vc];
      },
      [&](int u, long r) {
        bf16x8_t dr;
        put_to<PAST>((bf16x8_t*)(dx + r * C + m.vc * 8),
                     bn_dx<RELU, MASK>(p, mdb, mdw, ds[u], xs[u], ms[u], dr));
        if (dres) put_to<PAST>((bf16x8_t*)(dres + r * C + m.vc * 8), dr);
      });
}

// ---- few rows: a block has 16 channels (32 bytes of a row) and all rows,
// which its threads keep in registers between the sums and the result.
constexpr int SMALL = 512;             // threads
constexpr int COLS = 2;                // of 8 channels
constexpr int GROUPS = SMALL / COLS;   // rows at a time
constexpr int KEPT = 8;                // rows a thread keeps
constexpr long FEW = GROUPS * KEPT;

// s and q summed over the threads with the same columns, which all get the
// sums.  Lane l has column l % COLS.
DEVINL void small_sums(float (&s)[8], float (&q)[8],
                       float (&part)[SMALL / 16][COLS * 16],
                       float (&tot)[COLS * 16]) {
  const int t = threadIdx.x, c = t % COLS;
  auto strided = [](float v) {         // over every second of 16 lanes
    auto dpp = [](float x, auto ctrl) {
      return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
          0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v += dpp(v, std::integral_constant<int, 0x122>{});   // row_ror:2
    v += dpp(v, std::integral_constant<int, 0x124>{});   // row_ror:4
    v += dpp(v, std::integral_constant<int, 0x128>{});   // row_ror:8
    return v;
  };
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = strided(s[j]), b = strided(q[j]);
    if ((t & 15) < COLS) {
      part[t >> 4][c * 16 + j] = a;
      part[t >> 4][c * 16 + 8 + j] = b;
    }
  }
  __syncthreads();
  // 16 threads an entry, then the 16 lanes' sums
  const int e = t >> 4;
  if (e < COLS * 16) {
    float x = 0.f;
    #pragma unroll
    for (int w = 0; w < SMALL / 256; ++w) x += part[w * 16 + (t & 15)][e];
    #pragma unroll
    for (int o = 1; o < 16; o *= 2) x += __shfl_xor(x, o, 64);
    if ((t & 15) == 0) tot[e] = x;
  }
  __syncthreads();
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    s[j] = tot[c * 16 + j];
    q[j] = tot[c * 16 + 8 + j];
  }
}

template <bool RELU, bool RES>
__global__ void __launch_bounds__(SMALL)
bn_small_fwd_kernel(const short* __restrict__ x, const short* __restrict__ res,
                    const float* __restrict__ w, const float* __restrict__ b,
                    StatsOut o, short* __restrict__ y,
                    unsigned char* __restrict__ mask, int R, int C) {
  __shared__ float part[SMALL / 16][COLS * 16], tot[COLS * 16];
  // columns behind the last are the last once more, and are not stored
  const int mine = blockIdx.x * COLS + threadIdx.x % COLS;
  const int vc = min(mine, C / 8 - 1), g = threadIdx.x / COLS;
  const bool own = mine == vc;
  bf16x8_t xs[KEPT], rs[KEPT];
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {     // behind the last row: that one again
    const long at = (long)min(u * GROUPS + g, R - 1) * C + vc * 8;
    xs[u] = *(const bf16x8_t*)(x + at);
    if (RES) rs[u] = *(const bf16x8_t*)(res + at);
  }
  Channel8 p(vc, w, w, w, b);          // mean and 1/std follow
  float s[8] = {}, q[8] = {};
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {
    const bool in = u * GROUPS + g < R;
    const F8 xv = up8(xs[u]);
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] += in ? xv.v[j] : 0.f;
      q[j] += in ? xv.v[j] * xv.v[j] : 0.f;
    }
  }
  small_sums(s, q, part, tot);
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float mu = s[j] / (float)R, var = q[j] / (float)R - mu * mu;
    if (g == j && own) put_stats(o, vc * 8 + j, mu, var, R);
    p.mu[j] = mu;
    p.rs[j] = rsqrtf(fmaxf(var, 0.f) + o.eps);
  }
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {
    const int r = u * GROUPS + g;
    if (r >= R || !own) continue;
    unsigned bits;
    *(bf16x8_t*)(y + (long)r * C + vc * 8) = bn_out<RELU, RES>(p, xs[u], rs[u], bits);
    if (RELU && RES) mask[(long)r * (C / 8) + vc] = (unsigned char)bits;
  }
}

template <bool RELU, bool MASK>
__global__ void __launch_bounds__(SMALL)
bn_small_bwd_kernel(const short* __restrict__ dy, const short* __restrict__ x,
                    const unsigned char* __restrict__ mask,
                    const float* __restrict__ mean,
                    const float* __restrict__ rstd,
                    const float* __restrict__ w, const float* __restrict__ b,
                    float* __restrict__ dw, float* __restrict__ db,
                    short* __restrict__ dx, short* __restrict__ dres, int R,
                    int C) {
  __shared__ float part[SMALL / 16][COLS * 16], tot[COLS * 16];
  // columns behind the last are the last once more, and are not stored
  const int mine = blockIdx.x * COLS + threadIdx.x % COLS;
  const int vc = min(mine, C / 8 - 1), g = threadIdx.x / COLS;
  const bool own = mine == vc;
  bf16x8_t ds[KEPT], xs[KEPT];
  unsigned ms[KEPT];
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {
    const long r = min(u * GROUPS + g, R - 1);
    ds[u] = *(const bf16x8_t*)(dy + r * C + vc * 8);
    xs[u] = *(const bf16x8_t*)(x + r * C + vc * 8);
    if (MASK) ms[u] = mask[r * (C / 8) + vc];
  }
  const Channel8 p(vc, mean, rstd, w, b);
  float sd[8] = {}, sx[8] = {};
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {
    const bool in = u * GROUPS + g < R;
    float d[8], xh[8];
    bn_grad<RELU, MASK>(p, ds[u], xs[u], ms[u], d, xh);
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      sd[j] += in ? d[j] : 0.f;
      sx[j] += in ? d[j] * xh[j] : 0.f;
    }
  }
  small_sums(sd, sx, part, tot);
  const float invR = 1.f / (float)R;
  float mdb[8], mdw[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (g == j && own) {
      db[vc * 8 + j] = sd[j];
      dw[vc * 8 + j] = sx[j];
    }
    mdb[j] = sd[j] * invR;
    mdw[j] = sx[j] * invR;
  }
  #pragma unroll
  for (int u = 0; u < KEPT; ++u) {
    const int r = u * GROUPS + g;
    if (r >= R || !own) continue;
    bf16x8_t dr;
    *(bf16x8_t*)(dx + (long)r * C + vc * 8) =
        bn_dx<RELU, MASK>(p, mdb, mdw, ds[u], xs[u], ms[u], dr);
    if (dres) *(bf16x8_t*)(dres + (long)r * C + vc * 8) = dr;
  }
}

void check_nhwc(const torch::Tensor& t, const char* nm) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 4 &&
              t.is_contiguous(at::MemoryFormat::ChannelsLast), nm,
              " must be 4-D channels_last on the GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, nm, " must be bf16");
}

// a number for each channel
void check_channels(const torch::Tensor& t, int C, const char* nm) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 &&
              t.is_contiguous() && t.numel() == C, nm,
              " must be one float32 per channel, contiguous on the GPU");
}

dim3 row_grid(long R, int C, int ns) {
  const int CV = C / 8;
  return dim3(CV >= 256 ? (CV + 255) / 256 : 1, ns);
}

int slices(long R, int C) {
  // 8192 row streams, 8 (4) rows of each in flight, fill the chip; more
  // slices only grow the second stage (both directions of 256 x 256 x 56 x
  // 56: 512 slices 20 us more than 256, 1024 71 us)
  const int CV = C / 8;
  const int cvb = CV >= 256 ? (CV + 255) / 256 : 1;
  const int G = CV >= 256 ? 1 : 256 / CV;
  long want = 8192 / ((long)G * cvb);
  if (want > 256) want = 256;
  const long max_useful = (R + G - 1) / G;
  if (want > max_useful) want = max_useful;
  return (int)std::max<long>(1, want);
}

// The passes that only stream: four rows a thread, those of a block next to each
// other.  Blocks in flight then stay within some MB of each other, which memory
// serves faster than 2048 blocks that walk all rows with the whole grid's stride:
// 256 x 256 x 56 x 56, apply 217 -> 203 us, dx 354 -> 266 (6.3 TB/s); with 2 rows a
// thread both passes cost 2 us less and 1024 channels 7 more, with 8 rows 27 us more.
// Fewer rows a thread where that leaves few blocks.  A direction in us, walked (before) and
// with 4, 2 and 1 rows: 2500 rows of 128, backward 9.5, 11.0, 9.9 and 9.6; 16000 rows 14.1,
// 13.6, 13.3, 13.3; 12544 rows of 512, forward 19.1, 19.4, 18.7, 19.7; 32768 rows 30.7, 29.1,
// 29.2 and 30.8.  More where half the blocks have few channels: 50176 rows of 2056, walked and
// with 4 and 8, forward 243, 252 and 238, of 4096 25088 rows 163, 158 and 161.
struct Stream { dim3 grid; long span; };

Stream stream_grid(long R, int C) {
  const int CV = C / 8;
  const int cvb = CV >= 256 ? (CV + 255) / 256 : 1;
  const int G = CV >= 256 ? 1 : 256 / CV;
  const long ones = cvb * ((R + G - 1) / G);            // blocks of one row a thread
  const bool part = CV > 256 && CV % 256;               // a block of few threads at work
  const int rows = ones <= 1024 ? 1 : ones <= 3584 ? 2 : ones > 16384 && part ? 8 : 4;
  const long span = std::max<long>(rows * G, (R + 65534) / 65535);   // grid.y's limit
  return {dim3(cvb, (unsigned)((R + span - 1) / span)), span};
}

// Large results go past the caches, and so does the residual, which is read once: what the
// first pass has left in the memory-side cache of x and dy stays for the second, and the next
// first pass does not wait for lines to be written back.  Both directions in us, through the
// caches and past them, alone and with the results read once more behind it: 411 MB with a
// residual 728 and 657, 1126 and 1085, 206 MB 371 and 328, 584 and 559, 103 MB 186 and 167, 311
// and 289; but 51 MB without one 75 and 75, 111 and 113, 26 MB 49 and 48, 67 and 69.
bool past_caches(long R, int C) { return R * C >= 32l << 20; }

// One launch a direction instead of three, as long as a block's threads can
// keep their rows.  GPU time of forward + backward in us, one launch and three:
// 1568 rows of 512 channels 18.1 and 21.6, of 2048 29 and 36; 2048 rows of 512
// 19.3 and 21.7, 64 rows of 64 13.5 and 15.0; 2048 rows of 64, which are 4
// blocks, 18.3 and 17.4, against four launches less for the host.  At least one
// row: the kernels read the last one for lanes behind it.
bool few_rows(long R) { return R <= FEW; }

}  // namespace

// y = relu?(BN(x) [+ res]) in training mode; returns {y, mean, rstd}, and
// with both ReLU and res the bits of its sign, (N*H*W, C/8) bytes.
std::vector<torch::Tensor> bn_fwd(torch::Tensor x,
                                  c10::optional<torch::Tensor> res,
                                  torch::Tensor weight, torch::Tensor bias,
                                  c10::optional<torch::Tensor> running_mean,
                                  c10::optional<torch::Tensor> running_var,
                                  double momentum, double eps, bool relu) {
  CHECK_CUDA(x);
  check_nhwc(x, "x");
  const int C = (int)x.size(1);
  TORCH_CHECK(C > 0 && C % 8 == 0, "bn_fwd: C % 8 != 0");
  check_channels(weight, C, "weight");
  check_channels(bias, C, "bias");
  TORCH_CHECK(running_mean.has_value() == running_var.has_value(),
              "bn_fwd: one running statistic without the other");
  if (running_mean.has_value()) {
    check_channels(*running_mean, C, "running_mean");
    check_channels(*running_var, C, "running_var");
  }
  const long R = x.numel() / C;
  auto fopt = torch::TensorOptions().dtype(torch::kFloat32).device(x.device());
  auto mean = torch::empty({C}, fopt);
  auto rstd = torch::empty({C}, fopt);
  auto y = torch::empty_like(x);
  auto st = scaffold_stream();
  const short* rp = nullptr;
  torch::Tensor mask;
  unsigned char* mp = nullptr;
  if (res.has_value()) {
    check_nhwc(res.value(), "res");
    TORCH_CHECK(res->sizes() == x.sizes(), "bn_fwd: res must be as large as x");
    rp = (const short*)res->data_ptr();
    if (relu) {
      mask = torch::empty({R, C / 8}, fopt.dtype(torch::kUInt8));
      mp = mask.data_ptr<unsigned char>();
    }
  }
  if (R == 0) {                        // as torch: the statistics stay
    mean.zero_();
    rstd.zero_();
    if (mask.defined()) return {y, mean, rstd, mask};
    return {y, mean, rstd};
  }
  const StatsOut o{mean.data_ptr<float>(), rstd.data_ptr<float>(),
                   running_mean ? running_mean->data_ptr<float>() : nullptr,
                   running_var ? running_var->data_ptr<float>() : nullptr,
                   (float)momentum, (float)eps};
  const short* xp = (const short*)x.data_ptr();
  short* yp = (short*)y.data_ptr();
  const float *wp = weight.data_ptr<float>(), *bp = bias.data_ptr<float>();
  auto by_kind = [&](auto go) {
    using T = std::true_type;
    using F = std::false_type;
    if (relu && rp) go(T{}, T{});
    else if (relu) go(T{}, F{});
    else if (rp) go(F{}, T{});
    else go(F{}, F{});
  };
  if (few_rows(R)) {
    by_kind([&](auto rl, auto rs) {
      hipLaunchKernelGGL((bn_small_fwd_kernel<decltype(rl)::value, decltype(rs)::value>),
                         dim3((C / 8 + COLS - 1) / COLS), dim3(SMALL), 0, st, xp, rp, wp, bp, o,
                         yp, mp, (int)R, C);
    });
  } else {
    const int ns = slices(R, C);
    const Stream stream = stream_grid(R, C);
    auto mid = torch::empty({ns, 2, (long)C}, fopt);
    hipLaunchKernelGGL((bn_stats_kernel<8>), row_grid(R, C, ns), dim3(256), 0,
                       st, xp, mid.data_ptr<float>(), R, C);
    hipLaunchKernelGGL(bn_stats_final_kernel, dim3((C + 15) / 16), dim3(256),
                       0, st, mid.data_ptr<float>(), o, ns, R, C);
    by_kind([&](auto rl, auto rs) {
      constexpr bool RL = decltype(rl)::value, RS = decltype(rs)::value;
      auto* kernel = past_caches(R, C) ? &bn_apply_kernel<RL, RS, true>
                                       : &bn_apply_kernel<RL, RS, false>;
      hipLaunchKernelGGL(kernel, stream.grid, dim3(256), 0, st, xp, rp, o.mean,
                         o.rstd, wp, bp, yp, mp, R, C, stream.span);
    });
  }
  HIP_CHECK(hipGetLastError());
  if (mask.defined()) return {y, mean, rstd, mask};
  return {y, mean, rstd};
}

// {dx, dw, db}, or with a residual {dx, dres, dw, db}.  mask: what bn_fwd
// returned with both ReLU and a residual.
std::vector<torch::Tensor> bn_bwd(torch::Tensor dy, torch::Tensor x,
                                  bool has_res,
                                  c10::optional<torch::Tensor> mask,
                                  torch::Tensor weight, torch::Tensor bias,
                                  torch::Tensor mean, torch::Tensor rstd,
                                  bool relu) {
  CHECK_CUDA(dy);
  check_nhwc(x, "x");
  const int C = (int)x.size(1);
  TORCH_CHECK(C > 0 && C % 8 == 0, "bn_bwd: C % 8 != 0");
  check_channels(weight, C, "weight");
  check_channels(bias, C, "bias");
  check_channels(mean, C, "mean");
  check_channels(rstd, C, "rstd");
  const long R = x.numel() / C;
  TORCH_CHECK(mask.has_value() == (relu && has_res) &&
              (!mask.has_value() ||
               (mask->scalar_type() == torch::kUInt8 && mask->is_contiguous() &&
                mask->numel() == R * (C / 8))), "bn_bwd: mask");
  // as x lies: a slice of the channels and an expanded gradient have
  // stride(1) == 1 too
  TORCH_CHECK(dy.sizes() == x.sizes() && dy.scalar_type() == torch::kBFloat16,
              "bn_bwd: dy");
  auto dyc = dy.contiguous(at::MemoryFormat::ChannelsLast);
  auto fopt = torch::TensorOptions().dtype(torch::kFloat32).device(x.device());
  auto dw = torch::empty({C}, fopt);
  auto db = torch::empty({C}, fopt);
  auto dx = torch::empty_like(x);
  torch::Tensor dres;
  auto st = scaffold_stream();
  short* drp = nullptr;
  if (has_res) {
    dres = torch::empty_like(x);
    drp = (short*)dres.data_ptr();
  }
  if (R == 0) {
    dw.zero_();
    db.zero_();
    if (has_res) return {dx, dres, dw, db};
    return {dx, dw, db};
  }
  const unsigned char* mp = mask.has_value() ? mask->data_ptr<unsigned char>() : nullptr;
  const short *dp = (const short*)dyc.data_ptr(), *xp = (const short*)x.data_ptr();
  const float *mn = mean.data_ptr<float>(), *rs = rstd.data_ptr<float>();
  const float *wp = weight.data_ptr<float>(), *bp = bias.data_ptr<float>();
  float *dwp = dw.data_ptr<float>(), *dbp = db.data_ptr<float>();
  short* dxp = (short*)dx.data_ptr();
  auto by_kind = [&](auto go) {
    using T = std::true_type;
    using F = std::false_type;
    if (mp) go(T{}, T{});
    else if (relu) go(T{}, F{});
    else go(F{}, F{});
  };
  if (few_rows(R)) {
    by_kind([&](auto rl, auto mk) {
      hipLaunchKernelGGL((bn_small_bwd_kernel<decltype(rl)::value, decltype(mk)::value>),
                         dim3((C / 8 + COLS - 1) / COLS), dim3(SMALL), 0, st, dp, xp, mp, mn, rs,
                         wp, bp, dwp, dbp, dxp, drp, (int)R, C);
    });
  } else {
    const int ns = slices(R, C);
    const Stream stream = stream_grid(R, C);
    auto mid = torch::empty({ns, 2, (long)C}, fopt);
    by_kind([&](auto rl, auto mk) {
      hipLaunchKernelGGL((bn_bwd_reduce_kernel<decltype(rl)::value, decltype(mk)::value>),
                         row_grid(R, C, ns), dim3(256), 0, st, dp, xp, mp, mn,
                         rs, wp, bp, mid.data_ptr<float>(), R, C);
    });
    hipLaunchKernelGGL(bn_bwd_final_kernel, dim3((C + 15) / 16), dim3(256), 0,
                       st, mid.data_ptr<float>(), dwp, dbp, ns, C);
    by_kind([&](auto rl, auto mk) {
      constexpr bool RL = decltype(rl)::value, MK = decltype(mk)::value;
      auto* kernel = past_caches(R, C) ? &bn_bwd_dx_kernel<RL, MK, true>
                                       : &bn_bwd_dx_kernel<RL, MK, false>;
      hipLaunchKernelGGL(kernel, stream.grid, dim3(256), 0, st, dp, xp, mp, mn,
                         rs, wp, bp, dwp, dbp, dxp, drp, R, C, stream.span);
    });
  }
  HIP_CHECK(hipGetLastError());
  if (has_res) return {dx, dres, dw, db};
  return {dx, dw, db};
}

namespace {

// The node of batch_norm_act in the graph; issuing it from C++ is what few
// rows are bound by (32 x 512 x 7 x 7, both directions: 82 us from Python).
struct BatchNormAct : torch::autograd::Function<BatchNormAct> {
  using Ctx = torch::autograd::AutogradContext;
  static torch::Tensor forward(Ctx* ctx, torch::Tensor x,
                               c10::optional<torch::Tensor> res,
                               torch::Tensor weight, torch::Tensor bias,
                               c10::optional<torch::Tensor> running_mean,
                               c10::optional<torch::Tensor> running_var,
                               double momentum, double eps, bool relu) {
    at::AutoDispatchBelowADInplaceOrView guard;
    auto out = bn_fwd(x, res, weight, bias, running_mean, running_var,
                      momentum, eps, relu);
    ctx->save_for_backward({x, weight, bias, out[1], out[2],
                            out.size() > 3 ? out[3] : torch::Tensor()});
    ctx->saved_data["relu"] = relu;
    ctx->saved_data["res"] = res.has_value();
    return out[0];
  }
  static torch::autograd::variable_list backward(
      Ctx* ctx, torch::autograd::variable_list dy) {
    const auto s = ctx->get_saved_variables();
    const bool has_res = ctx->saved_data["res"].toBool();
    c10::optional<torch::Tensor> mask;
    if (s[5].defined()) mask = s[5];
    auto g = bn_bwd(dy[0], s[0], has_res, mask, s[1], s[2], s[3], s[4],
                    ctx->saved_data["relu"].toBool());
    const torch::Tensor none;
    return {g[0], has_res ? g[1] : none, g[has_res ? 2 : 1],
            g[has_res ? 3 : 2], none, none, none, none, none};
  }
};

}  // namespace

torch::Tensor batch_norm_act(torch::Tensor x, c10::optional<torch::Tensor> res,
                             torch::Tensor weight, torch::Tensor bias,
                             c10::optional<torch::Tensor> running_mean,
                             c10::optional<torch::Tensor> running_var,
                             double momentum, double eps, bool relu) {
  const auto nhwc = at::MemoryFormat::ChannelsLast;
  if (res.has_value()) res = res->contiguous(nhwc);
  return BatchNormAct::apply(x.contiguous(nhwc), res, weight, bias,
                             running_mean, running_var, momentum, eps, relu);
}
