// Device-side helpers shared by every gfx950 kernel (no torch headers, so
// kernel files with raw-pointer launchers compile in seconds).
// Target: MI355X only — wave64, 256 CUs / 8 XCDs, 160 KiB LDS/CU.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#define WAVE 64
#define DEVINL __device__ __forceinline__
#define INLINE __attribute__((always_inline))    // of lambdas

using bf16 = __hip_bfloat16;

// vector types for wide loads (G13: always vectorize bf16 as short4/short8)
typedef short bf16x4 __attribute__((ext_vector_type(4)));   // 8 B
typedef short bf16x8 __attribute__((ext_vector_type(8)));   // 16 B
typedef float f32x4 __attribute__((ext_vector_type(4)));    // 16 B
typedef float f32x16 __attribute__((ext_vector_type(16)));

DEVINL float bf2f(short u) {
  union { unsigned int i; float f; } c;
  c.i = ((unsigned int)(unsigned short)u) << 16;
  return c.f;
}

DEVINL short f2bf(float f) {
  // round-to-nearest-even bf16 conversion
  union { float f; unsigned int i; } c;
  c.f = f;
  unsigned int x = c.i;
  unsigned int rounded = x + 0x7FFF + ((x >> 16) & 1);
  if ((x & 0x7F800000u) == 0x7F800000u) rounded = x;  // inf/nan passthrough
  return (short)(rounded >> 16);
}

// Two float32 to a dword of two bf16, to nearest even: v_cvt_pk_bf16_f32.  Not
// in assembly, before which the compiler leaves out the wait that a result of
// v_exp_f32 needs.
DEVINL unsigned cvt_pk_bf16(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f2{lo, hi}), b2));
}

// f(0) ... f(N - 1), each number a constant
template <typename F, int... I>
DEVINL void each_of(const F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int N, typename F>
DEVINL void each(const F& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

// Past the caches, or through them: for what is read or written once in passes whose operands
// and results are together more than the memory-side cache holds, 256 MB, so that this keeps
// what will be asked for again, and does not have to write back before it takes something in.
template <bool PAST, typename V>
DEVINL void put_to(V* to, V v) {
  if constexpr (PAST) __builtin_nontemporal_store(v, to);
  else *to = v;
}
template <bool PAST, typename V>
DEVINL V get_from(const V* from) {
  if constexpr (PAST) return __builtin_nontemporal_load(from);
  else return *from;
}

// a value that is the same in all lanes, where the compiler does not see it (and
// would loop over the lanes to make a buffer descriptor of it)
DEVINL unsigned same(unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); }

// Bits 2 and 3 change places: score products of 32 x 32 whose rows are keys in this
// order leave a lane, in registers 8 i ..., the weights of consecutive keys.
DEVINL int swapped(int row) {
  return (row & ~12) | (row & 4) << 1 | (row & 8) >> 1;
}

// wave-level reductions (wave64)
DEVINL float wave_reduce_sum(float v) {
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

DEVINL float wave_reduce_max(float v) {
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// block reduction via LDS; `red` shared array must hold >= blockDim.x/64 floats
DEVINL float block_reduce_sum(float v, float* red) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  v = wave_reduce_sum(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  v = (lane < nwaves) ? red[lane] : 0.f;
  v = wave_reduce_sum(v);
  // broadcast through lane 0 of wave 0
  if (threadIdx.x == 0) red[0] = v;
  __syncthreads();
  float out = red[0];
  __syncthreads();
  return out;
}

DEVINL float block_reduce_max(float v, float* red) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  v = wave_reduce_max(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  v = (lane < nwaves) ? red[lane] : -INFINITY;
  v = wave_reduce_max(v);
  if (threadIdx.x == 0) red[0] = v;
  __syncthreads();
  float out = red[0];
  __syncthreads();
  return out;
}

// ---- 16 x 16 += 16 x 32 of a . (16 x 32 of b)^T
DEVINL f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// z Phi(z), with Phi(-t) = 2^P(t), t = |z|: P of degree 10, P(0) = -1, fitted on [0, 7] to the
// logarithm in 64 bits, weighted with Phi(-t), by least squares whose weights follow the
// largest error (Lawson's method); behind 7 it only falls, and 2^P(16) is 0.  Largest errors
// against 64 bits 5.6e-8 up to 1 and 2.4e-7 up to 12, where 0.5 z (1 + erff(z / sqrt 2)) has
// 8.5e-8 and 4.5e-7, and 5e-5 of the value down to -5, there 5 %.
DEVINL float gelu_erf(float z) {
  const float t = fminf(fabsf(z), 16.f);
  float p = -2.1855125709180358e-8f;
  p = fmaf(p, t, 7.03961745784909e-7f);
  p = fmaf(p, t, -9.565534128341824e-6f);
  p = fmaf(p, t, 6.97065843269229e-5f);
  p = fmaf(p, t, -2.606377238407731e-4f);
  p = fmaf(p, t, -3.2546609872952104e-5f);
  p = fmaf(p, t, 6.980439648032188e-3f);
  p = fmaf(p, t, -5.246090516448021e-2f);
  p = fmaf(p, t, -4.592151641845703e-1f);
  p = fmaf(p, t, -1.1511048078536987f);
  p = fmaf(p, t, -1.f);
  return fmaf(z > 0.f ? -t : z, __builtin_amdgcn_exp2f(p), fmaxf(z, 0.f));
}

// tanh(u) = 1 - 2 / (exp(2u) + 1), also at both ends.  The reciprocal with a Newton step,
// for which its operand stays finite: errors against 64 bits are those of a division to
// five digits (largest 9.4e-8 up to 1, 3.7e-7 up to 12), 1 % more without the step; a
// division at the end of a product of one row is 0.4 us of 4.3.
DEVINL float gelu_tanh(float z) {
  const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  const float d = __expf(fminf(2.f * u, 80.f)) + 1.f, r = __builtin_amdgcn_rcpf(d);
  return 0.5f * z * (2.f - 2.f * fmaf(fmaf(-d, r, 1.f), r, r));
}

// ---- LDS transpose-read machinery (guide T10, §2 "ds_read_b64_tr_b16")
//
// The tr-image of a [KT rows][D cols] bf16 tile packs 4x16 subtiles
// consecutively: element (k, d) lives at
//   el = ((k>>2) * (D/16) + (d>>4)) * 64 + (k&3)*16 + (d&15)
// written coalesced (16-aligned 8-element chunks).
//
// ds_read_b64_tr_b16 semantics — measured on hardware by probe_tr
// (benchmarks/tr_probe.py, 2026-09-13), NOT the guide's ambiguous
// wording: each lane reads 8 CONTIGUOUS bytes at its own 8-B-aligned
// address; within each 16-lane group the hardware then redistributes so
// lane l receives the bf16 at positions {16*j + (l&15), j=0..3} of the
// group's 64 concatenated elements (lane p's 4 els sit at positions
// 4p..4p+3).  To hand lane l column (l&15) of a [4 k-rows][16 d-cols]
// row-major subtile, lane p=(l&15) must therefore read
//   subtile_byte_base + (p>>2)*32 + (p&3)*8.

// async global->LDS copy, 16 B per lane (guide §5 common-mistake 1);
// dest is wave-uniform base + lane*16, source is per-lane.
DEVINL void glds16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)g,
      (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

DEVINL unsigned lds_byte_off(const void* p) {
  // generic -> LDS address space; uintptr of an AS(3) pointer is the
  // LDS byte offset the DS instructions take.
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// One transpose read at a byte offset into LDS.  The compiler schedules it and
// waits for as many as a matrix instruction needs: against batches behind one
// wait in assembly, training attention of 2 x 32 x 4096 x 128 took 609 us
// instead of 646 forward and 1305 instead of 1338 for dK and dV, prompt
// attention over pages 136 instead of 148 (with packed conversions).  The
// others, 1 x 4096 tokens or 64 rows at 4000, builtin and assembly in us: tied
// prompts 215 and 236, windows 99 and 106, latent prompts 91 and 92, latent
// decoding 37.2 and 38.0, tied decoding 55 and 55, states of retention 31.3 and
// 31.1, of Mamba-2 50.5 and 53.2, of gated linear attention 16.5 and 17.6, their
// outputs 54.7 and 55.8, 86.8 and 88.0, 32.3 and 32.1 (4 x 777: 31.7 and 31.2).
DEVINL bf16x4 tr_read(unsigned at) {
  typedef __attribute__((address_space(3))) bf16x4* P;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)at);
}

// two tr reads (k-quads q4 and q4+1) -> one bf16x8 A/B fragment in k-order
DEVINL bf16x8 tr_read_frag(unsigned addr_q0, unsigned addr_q1) {
  return __builtin_shufflevector(tr_read(addr_q0), tr_read(addr_q1), 0, 1, 2, 3,
                                 4, 5, 6, 7);
}

// A softmax weight as three bf16 parts whose sum it is, to float32's last bit: 8
// significand bits cut off at a time.  No part of a weight above zero is zero
// (the smallest normal number stands in), which would make an infinite value
// NaN.
struct WeightParts { short hi, mid, lo; };

DEVINL WeightParts weight_parts(float x) {
  auto bits = [](float y) { return __builtin_bit_cast(unsigned, y); };
  auto cut = [&](float y) { return __builtin_bit_cast(float, bits(y) & 0xffff0000u); };
  const float least = x > 0.f ? 1.1754943508222875e-38f : 0.f;
  const float y = fmaxf(x - cut(x), least), z = fmaxf(y - cut(y), least);
  return {(short)(bits(x) >> 16), (short)(bits(y) >> 16), (short)(bits(z) >> 16)};
}

struct bf16x8_quad { bf16x8 f[4]; };

DEVINL bf16x8_quad tr_read_quad(unsigned a0, unsigned a1, unsigned b0,
                                unsigned b1, unsigned c0, unsigned c1,
                                unsigned d0, unsigned d1) {
  return {{tr_read_frag(a0, a1), tr_read_frag(b0, b1), tr_read_frag(c0, c1),
           tr_read_frag(d0, d1)}};
}

struct bf16x8_pair { bf16x8 f[2]; };

DEVINL bf16x8_pair tr_read_pair(unsigned a0, unsigned a1, unsigned b0,
                                unsigned b1) {
  return {{tr_read_frag(a0, a1), tr_read_frag(b0, b1)}};
}

// XCD-affinity decomposition of a 1-D launch (guide T1): the dispatcher
// places block b on XCD b%8, so mapping every tile-block of one
// (batch, head) to ids ≡ bh (mod 8) co-locates them on ONE XCD — the
// K/V (fwd) or Q/dO (bwd) windows they all stage are then fetched from
// HBM once per chip instead of once per XCD (8x staging amplification
// measured as the dominant stall class of the bwd kernels).  Falls back
// to the identity map when 8 does not divide the bh count (speed-only
// either way — correctness never depends on placement).
DEVINL void xcd_tile_map(int nbx, int* bx, int* bh) {
  const unsigned id = blockIdx.x;
  const unsigned ubx = (unsigned)nbx;
  const unsigned gy = gridDim.x / ubx;
  if (gy % 8 == 0) {
    const unsigned xcd = id % 8, idx = id / 8;
    *bh = (int)(xcd + 8 * (idx / ubx));
    *bx = (int)(idx % ubx);
  } else {
    *bx = (int)(id % ubx);
    *bh = (int)(id / ubx);
  }
}

// The same for blocks of unequal length: all heads' blocks of one tile, then
// all of the next, so that the last to start are the shortest (with head after
// head the last head's longest blocks end alone: 2 x 32 x 4096 x 128 left 28 %
// of the compute units idle).  Heads that share keys and values go to one XCD.
DEVINL void head_tile_map(int nbx, int B, int H, int G, int* bx, int* b, int* h) {
  const unsigned heads = (unsigned)(B * H), rep = (unsigned)(H / G);
  const unsigned id = blockIdx.x;
  unsigned bh = id % heads;
  *bx = (int)(id / heads);
  if ((unsigned)(B * G) % 8 == 0) {
    const unsigned in = bh / 8;                    // of an XCD's heads
    const unsigned pair = bh % 8 + 8 * (in / rep);
    bh = pair * rep + in % rep;
  }
  *b = (int)(bh / H);
  *h = (int)(bh % H);
}

// Grid sizing guideline 11: cap grid, grid-stride the rest.
DEVINL long grid_stride() { return (long)gridDim.x * blockDim.x; }

inline int capped_blocks(long total_threads, int block = 256, int cap = 2048) {
  long b = (total_threads + block - 1) / block;
  return (int)std::min<long>(b, cap);
}
