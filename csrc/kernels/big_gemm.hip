// Large products on the matrix cores: where they are faster than a library's, and how
// they are split.  The kernel, and what bounds it: big_gemm.h.

#include <c10/core/DeviceGuard.h>

#include "../common.h"
#include "../plain.h"
#include "big_gemm.h"
#include "tile_gemm.h"

namespace {

constexpr long UNITS = 256;          // compute units, each with one block

long up(long a, long b) { return (a + b - 1) / b; }

// Results that the caches would not keep go past them: in us, through and past, 4096 x 28672
// x 4096 731 and 685, 8192 x 8192 x 8192 757 and 741, 16384 x 3072 x 768 64 and 68.
template <bool ACOL, bool BCOL, int NT, int ACT>
void launch(BigArgs a, hipStream_t st) {
  a.tiles = (unsigned)(up(a.M, 256) * up(a.N, 32 * NT));
  if (!a.am) a.am = a.M;
  if (!a.bn) a.bn = a.N;
  a.stream = 2l * a.M * a.N > 112l << 20;
  hipLaunchKernelGGL((big::gemm_kernel<ACOL, BCOL, NT, ACT>),
                     dim3(std::min<unsigned>(a.tiles, UNITS)), dim3(256), 0, st, a);
}

// Tiles of 256 x 256, or of 256 x 192 where these leave less of the chip idle: a round of
// them takes 0.82 of the time.  In us, 256 and 192 wide: x w^T, 16384 x 2304 x 768 62 and 51,
// 16384 x 768 x 3072 71 and 65, 8192 x 3072 x 2048 97 and 81, 8192 x 2048 x 2048 54 and 78.
double rounds(const BigArgs& a, int nt) {
  return (double)up(up(a.M, 256) * up(a.N, 32 * nt), UNITS) * (nt == 6 ? 0.82 : 1.);
}

int columns(const BigArgs& a) { return rounds(a, 6) < rounds(a, 8) ? 6 : 8; }

// the chip's part that full tiles take over that many rounds
double at_work(const BigArgs& a, double rounds) {
  return (double)a.M * (double)a.N / (65536. * UNITS * rounds);
}

BigArgs of(const TileArgs& t) {
  BigArgs a = {};
  a.a = t.x; a.b = t.w; a.bias = t.bias; a.y = t.y;
  a.lda = t.ldx; a.ldb = t.K; a.ldy = t.ldy;
  a.M = t.M; a.N = t.N; a.K = t.K;
  return a;
}

// columns of x w^T, whose lanes store as many as a block has products across
int width(const BigArgs& a) { return a.N % 24 ? 8 : columns(a); }

}  // namespace

// Where it is faster than a library on the whole: of 250 random sizes of 300 to 33000 rows the mean
// is 0.79 of the library's time, with the erf GELU, of 150, 0.83; one in twelve is slower, by 2 to
// 18 %, all of them with whole tiles of 128 columns, which a library is quick at (big_alone() leaves
// it most of those: deeper than 512, 56 of 400 were more than 2 % slower, and 15 of 300 still are, by
// up to 14 %, all whole across).  In us,
// library and this.  Shallow products, whose stores a library waits for: 16384 rows, 768 to
// 2304 69 and 53, to 3072 78 and 67; 9208 x 1656 x 512 35 and 20; 1152 x 28168 x 896 (0.64) 79
// and 74; but 8360 x 14088 x 128 83 and 92.  Deeper ones with tiles left over, for which 192
// columns or persistent blocks are better: 8192 x 3072 x 2048 91 and 82, 13360 x 2304 x 3072 246
// and 143, 5080 x 18216 x 3328 436 and 432; but full rounds, 8192 x 2048 x 2048, 51 and 54,
// and 10024 x 5752 x 6016 488 and 488.  With the erf GELU behind it a pass over memory is
// saved: 8192 x 8192 x 2048 244 and 221, 2032 x 8192 x 2048 69 and 61, 11728 x 8352 x 5888 (0.97)
// 0.92 of it, but 6152 x 7760 x 6784 (0.71) 1.02, 2064 x 4528 x 3072 (0.56) 1.05.
bool big_takes(const TileArgs& t, TileAct act) {
  const BigArgs a = of(t);
  if (act == TILE_GELU_TANH || t.M < 256 || t.N < 128 || t.N % 8 || t.K < 128 || t.K % 128 ||
      t.K > 1 << 22 || t.ldx % 8 || t.ldx < t.K || t.ldx > 1 << 22 || t.ldy % 8 ||
      t.ldy > 1 << 22 || ((size_t)t.x | (size_t)t.w | (size_t)t.y) % 16 || (size_t)t.bias % 2)
    return false;
  const double busy = at_work(a, rounds(a, width(a)));
  // With whole tiles, those are not taken whose mean is the library's: of 22 without a GELU, 1152 or
  // 1280 deep and below 0.78, 0.96 (9 slower); with one, of 33 deeper than 2048 and below 0.78,
  // 0.99, of 11 deeper than 4096 and above 0.95, 1.02.
  const bool whole = t.N % 128 == 0;
  if (act == TILE_GELU_ERF) {
    if (t.K <= 2048) return busy >= 0.62;
    if (whole) return t.K <= 8192 && busy >= 0.78 && (t.K <= 4096 || busy <= 0.95);
    return t.K <= 4096 ? busy >= 0.62 : t.K <= 8192 && busy >= 0.75;
  }
  if (t.K <= 1280) return t.K >= 256 && busy >= (whole && t.K > 1024 ? 0.78 : 0.6);
  return t.K <= 4096 && busy >= 0.72 && busy <= 0.97;
}

// Alone, without a GELU or a residual, tiles that are whole across, as the library's are, gain
// nothing in one round, nor, 1280 to 2048 deep, in two.  More than 512 deep, its time 1: of 39 sizes
// in one round 1.03 (in us, 15215 x 1024 x 1152 31 and 33, 6038 x 2304 x 2560 54 and 57), of 16 in two
// 1.00 (6383 x 4096 x 1664 71 and 79); but of 22 in two of other depths 0.94, of 107 in more 0.89, of
// 156 with columns left over 0.82, none slower, and of 60 with tiles of 192 columns 0.85, none slower.
bool big_alone(const TileArgs& t) {
  const BigArgs a = of(t);
  if (t.N % 256 || t.K <= 512 || width(a) == 6) return true;
  const double r = rounds(a, 8);
  return r > 2 || (r == 2 && (t.K <= 1280 || t.K > 2048));
}

void big_gemm(const TileArgs& t, TileAct act, hipStream_t st) {
  const BigArgs a = of(t);
  const int nt = width(a);
  if (act == TILE_GELU_ERF && nt == 6) launch<false, false, 6, BIG_GELU_ERF>(a, st);
  else if (act == TILE_GELU_ERF) launch<false, false, 8, BIG_GELU_ERF>(a, st);
  else if (nt == 6) launch<false, false, 6, BIG_NONE>(a, st);
  else launch<false, false, 8, BIG_NONE>(a, st);
}

// x w^T + b + res; None where big_takes() says no.  One rounding, as linear_fwd has it, or (last)
// two, as a product and a sum have, so that results are the same bits.  The residual comes in while
// the results are stored, where a pass of its own reads the product and writes it again.  Of 37
// sizes of 2336 to 65536 rows it takes, every one is faster.  In us, the product and a pass,
// tiles of 128 (linear_fwd, of up to 1024 columns and depths) and this: 16384 x 768 x 768 38, 41
// and 29, 65536 x 256 x 256 39, 30 and 27, 12288 x 1024 x 1024 42, 48 and 33; 16384 x 768 x 3072 85
// and 73, 8040 x 2920 x 256 49 and 36, 26104 x 1032 x 3200 179 and 162.
c10::optional<torch::Tensor> residual_linear(const torch::Tensor& x, const torch::Tensor& w,
                                             const c10::optional<torch::Tensor>& bias,
                                             const torch::Tensor& res, bool last) {
  if (watched() || !x.is_cuda()) return c10::nullopt;
  auto whole = [&](const torch::Tensor& t) {
    return plain(t, x.device()) && t.is_contiguous();
  };
  if (x.dim() < 2 || w.dim() != 2 || !whole(x) || !whole(w) || !whole(res) ||
      (bias && (!whole(*bias) || bias->dim() != 1 || bias->size(0) != w.size(0))) ||
      x.numel() == 0 || x.size(-1) != w.size(1) || w.size(0) >= 1 << 30 ||
      x.numel() / w.size(1) >= 1 << 30)
    return c10::nullopt;
  auto shape = x.sizes().vec();
  shape.back() = w.size(0);
  if (res.sizes() != c10::IntArrayRef(shape)) return c10::nullopt;
  TileArgs t = {};
  t.K = (int)w.size(1);
  t.N = (int)w.size(0);
  t.M = (int)(x.numel() / t.K);
  t.x = (const short*)x.data_ptr();
  t.w = (const short*)w.data_ptr();
  t.bias = bias ? (const short*)bias->data_ptr() : nullptr;
  t.ldx = t.K;
  t.ldy = t.N;
  if ((size_t)res.data_ptr() % 16 || t.K > BIG_DEPTH_OF_TRAINING || !big_takes(t, TILE_NONE))
    return c10::nullopt;
  const c10::DeviceGuard guard(x.device());
  auto y = torch::empty(shape, x.options());
  t.y = (short*)y.data_ptr();
  BigArgs a = of(t);
  a.res = (const short*)res.data_ptr();
  auto st = scaffold_stream();
  const bool wide = width(a) == 8;
  if (last && wide) launch<false, false, 8, BIG_RESIDUAL_LAST>(a, st);
  else if (last) launch<false, false, 6, BIG_RESIDUAL_LAST>(a, st);
  else if (wide) launch<false, false, 8, BIG_RESIDUAL>(a, st);
  else launch<false, false, 6, BIG_RESIDUAL>(a, st);
  HIP_CHECK(hipGetLastError());
  return y;
}

// dW[N][K] = sum over t of dY[t][N] X[t][K] where that is faster than a library's, else None:
// where tiles keep two thirds of the chip at work.  In us, library and this: 28672 x 4096 out
// of 8192 rows 1646 and 1272, of 500 176 and 106; 4096 x 4096 out of 8192 240 and 188; 6144 x
// 4096 out of 1000 66 and 52; but 608 x 12888 out of 11800 (0.60) 225 and 236.
//
// Sums run in the order of the library (hipBLASLt of ROCm 7, at Llama-3-8B's widths; another
// version or width may differ), and the gradients are the same bits, but where it splits
// the tiles of a last round.  Deep sums of few rounds whose last is half empty stay with it (up
// to 4096 rows deep it does not split them): 4096 x 14336 out of 8192 rows would take 721 instead
// of 982, but 5000 of its 59 million gradients are rounded otherwise, no nearer to 64 bits or
// farther, after which a step of AdamW leaves the next gradients 2 % apart, the most that bf16
// lets them.  (128256 x 4096, the head, of 31 rounds, 7361 and 5691: 5000 of 525 million, and 0.7 %.)
bool weight_grad_takes(long T, long N, long K) {
  if (T < 256 || T >= 1l << 30 || N < 256 || K < 256 || N % 8 || K % 8 || N > 1l << 22 ||
      K > 1l << 22)
    return false;
  BigArgs a = {};
  a.M = (int)N; a.N = (int)K;
  const long tiles = up(N, 256) * up(K, 256), last = tiles % UNITS;
  return at_work(a, rounds(a, 8)) >= 0.66 &&
         !(T > 4096 && tiles < 4 * UNITS && last > 0 && last <= UNITS / 2);
}

c10::optional<torch::Tensor> wide_weight_grad(const torch::Tensor& dy, const torch::Tensor& x) {
  if (watched() || !dy.is_cuda() || !plain(dy, dy.device()) || !plain(x, dy.device()) ||
      dy.dim() != 2 || x.dim() != 2 || dy.size(0) != x.size(0) || !dy.is_contiguous() ||
      !x.is_contiguous() || ((size_t)dy.data_ptr() | (size_t)x.data_ptr()) % 16)
    return c10::nullopt;
  const long T = x.size(0), N = dy.size(1), K = x.size(1);
  if (!weight_grad_takes(T, N, K)) return c10::nullopt;
  BigArgs a = {};
  a.a = (const short*)dy.data_ptr();
  a.b = (const short*)x.data_ptr();
  a.M = (int)N; a.N = (int)K; a.K = (int)T;
  a.lda = N; a.ldb = a.ldy = K;
  // the operands' device, whichever is current: torch's product goes by it too
  const c10::DeviceGuard guard(dy.device());
  auto dw = torch::empty({N, K}, x.options());
  a.y = (short*)dw.data_ptr();
  launch<true, true, 8, BIG_NONE>(a, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return dw;
}

// dX[M][K] = sum over n of dY[M][n] W[n][K] where that is faster than a library's, else None:
// where tiles keep 0.72 of the chip at work, of 150 sizes every one.  In us, library and this:
// 16384 rows, 768 from 3072 86 and 68, 3072 from 768 85 and 68, 8192 rows, 4096 from 28672 1400
// and 1302, 14336 from 4096 716 and 642; but 2000 rows, 4096 from 28672 (0.60) 394 and 472.
//
// Of Llama-3-8B's products, 4096 and more deep, that library was seen to split the last round of
// its tiles, of 256 x 256 whatever this one's are, at 6002 to 7800 rows, not up to 5120 nor at full
// rounds (8000 to 8192 rows): there this one's bits are the same.  Elsewhere it is left out: 10000
// of 30 million values rounded otherwise are 0.9 % of the first step's gradients, and 4 % of the
// next's.
bool input_grad_takes(long M, long N, long K) {
  if (M < 256 || M >= 1l << 30 || N < 128 || N % 128 || N > 1l << 22 || K < 256 || K % 8 ||
      K > 1l << 22)
    return false;
  BigArgs a = {};
  a.M = (int)M; a.N = (int)K;
  return at_work(a, rounds(a, columns(a))) >= 0.72 &&
         !(N > BIG_DEPTH_OF_TRAINING && M > 5120 && up(M, 256) * up(K, 256) % UNITS != 0);
}

c10::optional<torch::Tensor> input_grad(const torch::Tensor& dy, const torch::Tensor& w) {
  if (watched() || !dy.is_cuda() || !plain(dy, dy.device()) || !plain(w, dy.device()) ||
      dy.dim() != 2 || w.dim() != 2 || dy.size(1) != w.size(0) || !dy.is_contiguous() ||
      !w.is_contiguous() || ((size_t)dy.data_ptr() | (size_t)w.data_ptr()) % 16)
    return c10::nullopt;
  const long M = dy.size(0), N = w.size(0), K = w.size(1);
  if (!input_grad_takes(M, N, K)) return c10::nullopt;
  BigArgs a = {};
  a.a = (const short*)dy.data_ptr();
  a.b = (const short*)w.data_ptr();
  a.M = (int)M; a.N = (int)K; a.K = (int)N;
  a.lda = N; a.ldb = a.ldy = K;
  const c10::DeviceGuard guard(dy.device());
  auto dx = torch::empty({M, K}, dy.options());
  a.y = (short*)dx.data_ptr();
  if (columns(a) == 6) launch<false, true, 6, BIG_NONE>(a, scaffold_stream());
  else launch<false, true, 8, BIG_NONE>(a, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return dx;
}

// The head of a language model whose vocabulary is no multiple of eight: rows of logits and of
// their gradients, 16 bytes apart at odd places, are what a library reads and writes slowly.
// Here they lie in rows of whole lines.  In us, library with rows of 50257 and this: 16384
// rows of 768, logits 1154 and 1001, dx 1203 and 989, dW 1352 and 1031.
//
// x (R, K) w (V, K)^T, as (R, V) with rows of V rounded up to 128; None where it is not for that.
c10::optional<torch::Tensor> head_logits(const torch::Tensor& x, const torch::Tensor& w) {
  if (watched() || !x.is_cuda() || !plain(x.detach(), x.device()) ||
      !plain(w.detach(), x.device()) || x.dim() != 2 || w.dim() != 2 ||
      x.size(1) != w.size(1) || !x.is_contiguous() || !w.is_contiguous())
    return c10::nullopt;
  const long V = w.size(0), K = w.size(1), R = x.size(0), ld = up(V, 128) * 128;
  if (V % 8 == 0 || V >= 1l << 22 || R >= 1l << 30) return c10::nullopt;
  TileArgs t = {};
  t.x = (const short*)x.data_ptr();
  t.w = (const short*)w.data_ptr();
  t.M = (int)R; t.N = (int)(up(V, 8) * 8); t.K = (int)K;
  t.ldx = K; t.ldy = ld;
  if (!big_takes(t, TILE_NONE)) return c10::nullopt;
  const c10::DeviceGuard guard(x.device());
  auto y = torch::empty({R, ld}, x.options());
  t.y = (short*)y.data_ptr();
  BigArgs a = of(t);
  a.bn = (int)V;
  if (width(a) == 6) launch<false, false, 6, BIG_NONE>(a, scaffold_stream());
  else launch<false, false, 8, BIG_NONE>(a, scaffold_stream());
  HIP_CHECK(hipGetLastError());
  return y.narrow(1, 0, V);
}

// {d w, d^T x} of such logits' gradient d, zero behind its last column; undefined where not
// wanted.  By torch where the rows lie otherwise: a saved tensor that a hook has copied comes
// back with one row behind the other.
std::vector<torch::Tensor> head_grads(const torch::Tensor& d, const torch::Tensor& x,
                                      const torch::Tensor& w, bool want_x, bool want_w) {
  auto whole = [&](const torch::Tensor& t) {
    return plain(t, d.device()) && t.dim() == 2 && t.is_contiguous() &&
           (size_t)t.data_ptr() % 16 == 0;
  };
  if (watched() || !d.is_cuda() || !plain(d, d.device()) || d.dim() != 2 || !whole(x) ||
      !whole(w) || x.size(0) != d.size(0) || w.size(0) != d.size(1) || x.size(1) != w.size(1) ||
      x.size(1) % 8 || d.stride(1) != 1 || d.stride(0) != up(d.size(1), 128) * 128 ||
      d.storage_offset() != 0 || (long)d.storage().nbytes() < 2 * d.size(0) * d.stride(0) ||
      (size_t)d.data_ptr() % 16)
    return {want_x ? at::mm(d, w) : torch::Tensor(), want_w ? at::mm(d.t(), x) : torch::Tensor()};
  const long R = d.size(0), V = w.size(0), K = w.size(1), ld = d.stride(0);
  const c10::DeviceGuard guard(d.device());
  auto st = scaffold_stream();
  torch::Tensor dx, dw;
  BigArgs a = {};
  a.a = (const short*)d.data_ptr();
  a.lda = ld;
  if (want_x) {
    a.b = (const short*)w.data_ptr();
    a.M = (int)R; a.N = (int)K; a.K = (int)V;
    a.ldb = a.ldy = K;
    const int nt = columns(a);
    if (at_work(a, rounds(a, nt)) >= 0.72) {
      dx = torch::empty({R, K}, x.options());
      a.y = (short*)dx.data_ptr();
      if (nt == 6) launch<false, true, 6, BIG_NONE>(a, st);
      else launch<false, true, 8, BIG_NONE>(a, st);
    } else {
      dx = at::mm(d, w);
    }
  }
  if (want_w) {
    a.b = (const short*)x.data_ptr();
    a.M = (int)V; a.N = (int)K; a.K = (int)R;
    a.am = (int)ld; a.bn = 0;
    a.ldb = a.ldy = K;
    if (at_work(a, rounds(a, 8)) >= 0.66) {
      dw = torch::empty({V, K}, w.options());
      a.y = (short*)dw.data_ptr();
      launch<true, true, 8, BIG_NONE>(a, st);
    } else {
      dw = at::mm(d.t(), x);
    }
  }
  HIP_CHECK(hipGetLastError());
  return {dx, dw};
}
