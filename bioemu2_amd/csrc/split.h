// fp32 products on the f16 matrix cores, for gfx950.
//
// An fp32 value x, scaled by a power of two, is carried as two f16 values
//   hi = f16(x),  lo = f16(x - hi)          (22-24 significant bits together)
// and a product of two such operands as three f16 MFMAs with fp32
// accumulation: lo*hi + hi*lo + hi*hi (lo*lo is below half an ulp of x*y).
// v_mfma_f32_32x32x16_f16 does 16 k in 32 cycles against 8 x 64 cycles of
// v_mfma_f32_32x32x2_f32, so the three cost 96 cycles where the fp32 MFMA
// takes 512.  Against float64 the result is at least as close as the fp32
// MFMA's for K >= 64, because it rounds its accumulator K / 16 * 3 times
// instead of K / 2 (relative error of a 32 x 32 block of normal data, measured:
// K = 64 1.15e-7 vs 1.49e-7, K = 128 1.47e-7 vs 1.89e-7, K = 384 2.3e-7 vs
// 3.5e-7, K = 1024 3.8e-7 vs 5.8e-7; K = 32 is a tie: attention's logits, K = 24
// and 32, and transitions of fewer than 64 channels or hidden units gain time
// only, and one product alone has up to twice the error of its fp32 form).
//
// Range: the scale brings the largest magnitude of a row (of activations or of
// weights) into [2^14, 2^15).  hi + lo is then exact to 2^-23 relative for
// elements down to 2^-16 of that maximum and to 2^-39 of the maximum below it
// (the f16 MFMA multiplies subnormals).  A scale depends on its own row (or on
// the weights) alone, so a row's result never depends on another row, nor an
// output channel's error on another channel's weights.  What a scale does not
// reach: inside one row, elements below 2^-16 of the row's largest keep fewer
// bits than fp32, which shows where the others' weights are that much smaller (a
// channel 1e5, 1e6, 1e7 times the rest under zero weights, through a whole
// transition: 2e-7, 8e-7, 1.3e-5; fp32 operands: 4e-7).  The same holds for a
// row's hidden values (per 32 of them, or up to the largest so far) and for 32
// keys' K and V of a head.  An infinite operand has no second part: its products
// are no numbers, where fp32 gives infinities (hidden values excepted).
//
// Operand fragments: 32 rows x 16 k are 1 KB of hi followed by 1 KB of lo,
// lane (n, h) = 8 consecutive values, row n, k = 8 h .. 8 h + 7.  Weight rows
// are stored in perm32 order (pairtile.h), so an accumulator lane ends with 16
// consecutive output channels of one activation row.
#pragma once

#include "common.h"
#include "internal.h"
#include "pairtile.h"

namespace bioemu {

typedef _Float16 f16;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kFragHalf = 512;         // f16 elements of one 32 x 16 plane (hi or lo): 1 KB
constexpr int kFrag = 2 * kFragHalf;   // hi | lo

struct SplitFrag {
  f16x8 hi, lo;
};

__device__ __forceinline__ f32x16 mfma_f16(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void mfma_split(const SplitFrag& a, const SplitFrag& b, f32x16& acc) {
  acc = mfma_f16(a.lo, b.hi, acc);
  acc = mfma_f16(a.hi, b.lo, acc);
  acc = mfma_f16(a.hi, b.hi, acc);
}

// 2^(14 - floor(log2 amax)), limited to 2^100 (amax = 0 or below 2^-86).
__device__ __forceinline__ float split_scale(float amax) {
  const int f = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xffu);
  return __builtin_bit_cast(float, (uint32_t)min(268 - f, 227) << 23);
}
// 1 / s of a power of two s from split_scale (exact).
__device__ __forceinline__ float split_inv(float s) {
  return __builtin_bit_cast(float, (uint32_t)(254 - (int)(__builtin_bit_cast(uint32_t, s) >> 23)) << 23);
}

// The larger of x in lanes l and l ^ 32: the halves exchanged by one VALU instruction instead of a trip through LDS.
__device__ __forceinline__ float max_halves(float x) {
  const unsigned b = __builtin_bit_cast(unsigned, x);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}

// x * s as hi + lo.  s is a power of two: the compiler may round the product to f16 in one step for hi and in two
// steps (through f32) for the hi that lo is taken from, and only an exact product makes both the same value.
__device__ __forceinline__ void split_value(float x, float s, f16& hi, f16& lo) {
  hi = (f16)(x * s);
  lo = (f16)__builtin_fmaf(x, s, -(float)hi);
}

// An infinite value as the largest finite one (its lo would be no number); the product overflows again.
__device__ __forceinline__ float split_finite(float x) {
  return (__builtin_bit_cast(uint32_t, x) & 0x7fffffffu) == 0x7f800000u ? __builtin_copysignf(3.40282347e38f, x) : x;
}

// log2(e) less its float value: the second part of a two-part constant.
constexpr float kLog2eLow = (float)(1.4426950408889634074 - (double)kLog2e);

// sigmoid(x) to about an ulp: the hardware exp2 on -x log2(e) carried as a rounded product and its error (the product of
// the two-part constant by fused multiply-adds; a plain product would cost |x| 2^-24 relative), and one Newton step on
// the hardware reciprocal.  Past +-87 the result is 1
// or 2e-38, where an infinite x would make the product's error and the Newton step NaN; the clamp drops a NaN x, which
// the last select returns (on its bits: the build lets the compiler fold x != x).
__device__ __forceinline__ float sigmoid_ulp(float x) {
  const float y = -fminf(fmaxf(x, -87.f), 87.f);
  const float t = y * kLog2e;
  const float r = __builtin_fmaf(y, kLog2eLow, __builtin_fmaf(y, kLog2e, -t));
  float e = fast_exp2(t);
  e = __builtin_fmaf(e, r * 0.6931471805599453f, e);
  const float d = 1.0f + e, q = fast_rcp(d);
  const float v = __builtin_fmaf(__builtin_fmaf(-d, q, 1.0f), q, q);
  return (__builtin_bit_cast(uint32_t, x) & 0x7fffffffu) > 0x7f800000u ? x : v;
}

__device__ __forceinline__ SplitFrag load_frag(const f16* p, int lane) {
  SplitFrag f;
  f.hi = *reinterpret_cast<const f16x8*>(p + lane * 8);
  f.lo = *reinterpret_cast<const f16x8*>(p + kFragHalf + lane * 8);
  return f;
}

// acc += the product of a 32 x 16 KS weight block (fragments in LDS at w) with xf; kWeightRows: the weights are the
// MFMA rows.  Two k-steps' fragments are in flight ahead of the one multiplied.
template <int KS, bool kWeightRows = true>
__device__ __forceinline__ void mfma_block(const f16* w, const SplitFrag* xf, int lane, f32x16& acc) {
  SplitFrag f[3];
  f[0] = load_frag(w, lane);
  f[1] = load_frag(w + kFrag, lane);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (s + 2 < KS) f[(s + 2) % 3] = load_frag(w + (s + 2) * kFrag, lane);
    __builtin_amdgcn_sched_barrier(0);
    if (kWeightRows)
      mfma_split(f[s % 3], xf[s], acc);
    else
      mfma_split(xf[s], f[s % 3], acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}
// Two weight blocks and two accumulators, a k-step of each at a time.
template <int KS, bool kWeightRows = true>
__device__ __forceinline__ void mfma_block2(const f16* w1, const f16* w2, const SplitFrag* x1, const SplitFrag* x2,
                                            int lane, f32x16& acc1, f32x16& acc2) {
  SplitFrag f1[2], f2[2];
  f1[0] = load_frag(w1, lane);
  f2[0] = load_frag(w2, lane);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (s + 1 < KS) {
      f1[(s + 1) & 1] = load_frag(w1 + (s + 1) * kFrag, lane);
      f2[(s + 1) & 1] = load_frag(w2 + (s + 1) * kFrag, lane);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kWeightRows) {
      mfma_split(f1[s & 1], x1[s], acc1);
      mfma_split(f2[s & 1], x2[s], acc2);
    } else {
      mfma_split(x1[s], f1[s & 1], acc1);
      mfma_split(x2[s], f2[s & 1], acc2);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ void copy1k_to_lds(__amdgpu_buffer_rsrc_t r, const f16* lds, unsigned voff, unsigned soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(lds), 16, voff, soff, 0, 0);
}

// ---------------------------------------------------------------------------
// Host side (split_gemm.hip).
// ---------------------------------------------------------------------------
// One weight matrix [rows][K] fp32 (K % 8 == 0; rows past the last are zeros) to fragments.  The block of
// rows 32 rb .. and the k-step ks (16 columns, zero past K) go to
//   dst + rb * rb_stride + (ks / kgrp) * kgrp_stride + (ks % kgrp) * kFrag
// for ks < ksteps; inv[32 rb * inv_stride + i] = 1 / scale of row 32 rb + i (rows past the
// last too) and, unless null, norm[32 rb * inv_stride + i] bounds |row . x| / |x| (its 2-norm).
//
// With gamma, a preceding LayerNorm's affine is folded in, so that rows are only
// centred and divided by their deviation: the fragments hold W diag(gamma),
// bias[row] = W beta (fp32; zero when beta is null) and norm bounds |W LN(x)|.
struct SplitMat {
  const float* w;
  f16* dst;
  float* inv;
  float* norm;
  int rows, K, ksteps, kgrp;
  long long rb_stride, kgrp_stride;
  int inv_stride;
  const float *gamma, *beta;
  float* bias;
};
constexpr int kSplitMats = 4;
struct SplitMats {
  SplitMat m[kSplitMats];
  int block_end[kSplitMats];   // set by split_prep
  void* zero;                  // split_weights: memory to clear, 16-byte aligned, a multiple of 16 bytes
  size_t zero_bytes;
};
// M rows x [M][K] fp32 (K % 8 == 0, 16-byte aligned), LayerNormed (biased variance, eps 1e-5) when g, to fragments;
// inv[row] = 1 / scale.
struct SplitRows {
  const float* x;
  const float *g, *b;
  f16* dst;
  float* inv;
  long long M;
  int K, ksteps;   // ksteps set by split_prep
};
int split_weights(const SplitMats& mats, int count, hipStream_t stream);
// count weights (0: none) and rows.
int split_prep(SplitMats mats, int count, SplitRows rows, hipStream_t stream);

// k-steps of a GEMM operand of K columns: whole pairs of 16 (the tile loop stages two at a time).
inline int split_ksteps(int64_t K) { return (int)(round_up(K, 32) / 16); }
// Bytes of the fragments of `rows` x K (rows rounded up to 32).
inline size_t split_frag_bytes(int64_t rows, int64_t K) {
  return (size_t)(round_up(rows, 32) / 32) * split_ksteps(K) * kFrag * sizeof(f16);
}

// A plain GEMM weight: row blocks in order (stride 1) or interleaved with a
// second matrix's (SwiGLU: fc1 blocks at even positions, fc2 at odd).
inline SplitMat split_gemm_weight(const float* w, f16* dst, float* inv, float* norm, int64_t rows, int64_t K,
                                  int interleave = 1, int first = 0) {
  const int ks = split_ksteps(K);
  return SplitMat{w, dst + (size_t)first * ks * kFrag, inv + 32 * first, norm ? norm + 32 * first : nullptr, (int)rows,
                  (int)K, ks, ks, (long long)interleave * ks * kFrag, 0, interleave, nullptr, nullptr, nullptr};
}
// With a LayerNorm's affine folded in.
inline SplitMat with_fold(SplitMat m, const float* gamma, const float* beta, float* bias) {
  m.gamma = gamma;
  m.beta = beta;
  m.bias = bias;
  return m;
}

}  // namespace bioemu
