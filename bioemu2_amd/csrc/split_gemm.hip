// GEMMs of the fp32 path on split f16 operands (split.h): out = epi(A W^T).
//
//   split_weights_kernel  weights -> fragments, once per call (a workgroup per
//                         block of 32 rows).
//   split_prep_kernel     the same and activation rows -> fragments, with the
//                         LayerNorm that precedes the product: a workgroup per 32
//                         rows of either, its four waves sharing the k-steps,
//                         statistics through LDS.
//   split_gemm_kernel     128 x 128 output tiles, 4 waves of 64 x 64; both operands
//                         staged through LDS two k-steps at a time by copies that
//                         write LDS directly (fragments are contiguous: no swizzle,
//                         no bank conflicts), double-buffered.
//   split_gemm_small_kernel  32 x 64 output tiles, the four waves of a workgroup
//                         splitting the k-steps: for row counts that would leave
//                         most CUs without a 128 x 128 tile.
//   split_gemm_r128_kernel  rows of 128 channels straight from fp32.
//
// Measured on the denoiser's shapes, against the fp32-MFMA kernels (operands from L2,
// a wave per 32 x 32 block) these replace: q, k, v, g of 6144 rows, K = 384, 0.131 ->
// 0.041 ms (178 TFLOP/s of fp32 products); of 49152 rows, K = 128, 0.127 -> 0.046 ms
// (125 MB, bound by its stores); output projections 0.039 -> 0.018 and 0.032 -> 0.019;
// 200 rows, K = 384 and 768 (small kernel): 0.023 -> 0.007 and 0.028 -> 0.008 ms.  The
// tiled kernel is bound by LDS: 8 fragment reads and 8 staged KB per 12 MFMAs.
#include <algorithm>

#include "split.h"
#include "split_gemm.h"
#include "split_rows.h"

namespace bioemu {
namespace {

// A workgroup per block of 32 rows; its waves share the k-steps.  What fits in kWaves x kSteps k-steps is read once,
// with every load in flight; longer weights are read again for the second pass.
constexpr int kSwWaves = 16, kSwSteps = 4;

// Columns k .. k + 7 of a row, times gamma; dot += the columns' product with beta.
__device__ __forceinline__ void weight_chunk(const SplitMat& m, const float* row, int k, int K, float (&v)[8],
                                             float& dot) {
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, c = a;
  if (k < K) {   // K is a multiple of 8
    a = *reinterpret_cast<const f32x4*>(row + k);
    c = *reinterpret_cast<const f32x4*>(row + k + 4);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    v[t] = a[t];
    v[4 + t] = c[t];
  }
  if (m.gamma && k < K) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if (m.beta) dot += v[t] * m.beta[k + t];
      v[t] *= m.gamma[k + t];
    }
  }
}

template <int kWaves, int kSteps>
__device__ __forceinline__ void split_weight_block(const SplitMat& m, int rb) {
  __shared__ float rowm[kWaves][32], rown[kWaves][32], rowd[kWaves][32];
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int r = rb * 32 + perm32(n), K = r < m.rows ? m.K : 0;   // rows past the matrix read as zeros
  const float* row = m.w + (size_t)r * m.K;
  float v[kSteps][8];
  float amax = 0.f, ss = 0.f, dot = 0.f, unused = 0.f;
#pragma unroll
  for (int i = 0; i < kSteps; ++i) weight_chunk(m, row, (wave + kWaves * i) * 16 + 8 * h, K, v[i], dot);
  auto scan = [&](const float (&c)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      amax = fmaxf(amax, fabsf(c[t]));
      ss += c[t] * c[t];
    }
  };
#pragma unroll
  for (int i = 0; i < kSteps; ++i) scan(v[i]);
  for (int ks = wave + kWaves * kSteps; ks < m.ksteps; ks += kWaves) {
    float c[8];
    weight_chunk(m, row, ks * 16 + 8 * h, K, c, dot);
    scan(c);
  }
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  ss += __shfl_xor(ss, 32);
  dot += __shfl_xor(dot, 32);
  if (lane < 32) {
    rowm[wave][lane] = amax;
    rown[wave][lane] = ss;
    rowd[wave][lane] = dot;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) amax = fmaxf(amax, rowm[w][n]);
  const float s = split_scale(amax);
  const size_t at = (size_t)rb * 32 * m.inv_stride + perm32(n);
  if (threadIdx.x < 32) m.inv[at] = split_inv(s);
  if (wave == 0 && (m.norm || m.bias)) {
    float q = 0.f, d = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      q += rown[w][n];
      d += rowd[w][n];
    }
    if (m.bias && lane < 32 && r < m.rows) m.bias[r] = d;
    // |x| <= sqrt(K) for a normalised row
    q = m.gamma ? sqrtf(q * (float)m.K) + fabsf(d) : sqrtf(q);
    if (m.norm && lane < 32) m.norm[at] = q;
  }
  auto put = [&](int ks, const float (&c)[8]) {
    f16x8 hi, lo;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      f16 a, b;
      split_value(c[t], s, a, b);
      hi[t] = a;
      lo[t] = b;
    }
    f16* d = m.dst + rb * m.rb_stride + (long long)(ks / m.kgrp) * m.kgrp_stride + (long long)(ks % m.kgrp) * kFrag;
    *reinterpret_cast<f16x8*>(d + lane * 8) = hi;
    *reinterpret_cast<f16x8*>(d + kFragHalf + lane * 8) = lo;
  };
#pragma unroll
  for (int i = 0; i < kSteps; ++i)
    if (wave + kWaves * i < m.ksteps) put(wave + kWaves * i, v[i]);
  for (int ks = wave + kWaves * kSteps; ks < m.ksteps; ks += kWaves) {
    float c[8];
    weight_chunk(m, row, ks * 16 + 8 * h, K, c, unused);
    put(ks, c);
  }
}

__global__ __launch_bounds__(64 * kSwWaves) void split_weights_kernel(SplitMats mats, int count) {
  if ((int)blockIdx.y == count) {
    uint4* p = static_cast<uint4*>(mats.zero);
    const size_t step = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < mats.zero_bytes / 16; i += step)
      p[i] = uint4{0, 0, 0, 0};
    return;
  }
  const SplitMat& m = mats.m[blockIdx.y];
  if ((int)blockIdx.x * 32 >= m.rows) return;   // uniform over the workgroup
  split_weight_block<kSwWaves, kSwSteps>(m, blockIdx.x);
}

// Sum over the row's two lanes and the workgroup's four waves (one value per row).
__device__ __forceinline__ float rows_sum(float v, float (&buf)[4][32], int wave, int lane) {
  v += __shfl_xor(v, 32);
  if (lane < 32) buf[wave][lane] = v;
  __syncthreads();
  const int n = lane & 31;
  return buf[0][n] + buf[1][n] + buf[2][n] + buf[3][n];
}
__device__ __forceinline__ float rows_max(float v, float (&buf)[4][32], int wave, int lane) {
  v = fmaxf(v, __shfl_xor(v, 32));
  if (lane < 32) buf[wave][lane] = v;
  __syncthreads();
  const int n = lane & 31;
  return fmaxf(fmaxf(buf[0][n], buf[1][n]), fmaxf(buf[2][n], buf[3][n]));
}

// Rows of K values (a multiple of 8), optionally LayerNormed (biased variance, eps
// 1e-5, fp32, two passes), to fragments.  A lane holds KPW k-steps x 8 values in
// registers; wave w takes the k-steps w, w + 4, ...  inv[row] = 1 / scale.
template <int KPW, bool kLn>
__device__ __forceinline__ void split_row_block(const SplitRows& r, long long rb) {
  __shared__ float buf[3][4][32];
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const long long m = rb * 32 + n, M = r.M;
  const bool valid = m < M;
  const int K = r.K, ksteps = r.ksteps;
  const float *g = r.g, *b = r.b;
  f16* dst = r.dst;
  float* inv = r.inv;
  float v[KPW][8];
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int k = (wave + 4 * i) * 16 + 8 * h;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, c = a;
    if (valid && k < K) {
      const float* p = r.x + (size_t)m * K + k;
      a = *reinterpret_cast<const f32x4*>(p);
      c = *reinterpret_cast<const f32x4*>(p + 4);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      v[i][t] = a[t];
      v[i][4 + t] = c[t];
    }
  }
  if (kLn) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < KPW; ++i)
#pragma unroll
      for (int t = 0; t < 8; ++t) s += v[i][t];
    const float mean = rows_sum(s, buf[0], wave, lane) / (float)K;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < KPW; ++i) {
      const int k = (wave + 4 * i) * 16 + 8 * h;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        v[i][t] = k < K ? v[i][t] - mean : 0.f;
        ss += v[i][t] * v[i][t];
      }
    }
    const float rstd = 1.0f / sqrtf(rows_sum(ss, buf[1], wave, lane) / (float)K + 1e-5f);
#pragma unroll
    for (int i = 0; i < KPW; ++i) {
      const int k = (wave + 4 * i) * 16 + 8 * h;
      if (k < K) {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[i][t] = v[i][t] * rstd * g[k + t] + (b ? b[k + t] : 0.f);
      }
    }
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < KPW; ++i)
#pragma unroll
    for (int t = 0; t < 8; ++t) amax = fmaxf(amax, fabsf(v[i][t]));
  amax = rows_max(amax, buf[2], wave, lane);
  const float s = split_scale(amax);
  if (wave == 0 && lane < 32 && valid) inv[m] = split_inv(s);
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int ks = wave + 4 * i;
    if (ks < ksteps) {
      f16x8 hi, lo;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f16 a, c;
        split_value(v[i][t], s, a, c);
        hi[t] = a;
        lo[t] = c;
      }
      f16* d = dst + ((size_t)rb * ksteps + ks) * kFrag;
      *reinterpret_cast<f16x8*>(d + lane * 8) = hi;
      *reinterpret_cast<f16x8*>(d + kFragHalf + lane * 8) = lo;
    }
  }
}

// Weight blocks (mats.m[i] holding block_end[i - 1] .. block_end[i]) and row blocks in one launch: neither depends on
// the other, and each alone is a chain of dependent memory round trips rather than bandwidth.  Two launches -> one at
// K = 384 and 768: 200 rows 14.3 -> 9.4 us, 6144 rows 17.4 -> 10.7 us.
template <int KPW, bool kLn>
__global__ __launch_bounds__(256) void split_prep_kernel(SplitMats mats, SplitRows rows) {
  const int blk = blockIdx.x;
  if (blk < mats.block_end[kSplitMats - 1]) {   // uniform over the workgroup
    int i = 0;
    while (blk >= mats.block_end[i]) ++i;
    const int rb = blk - (i ? mats.block_end[i - 1] : 0);
    if (mats.m[i].ksteps <= 4 * 6)
      split_weight_block<4, 6>(mats.m[i], rb);
    else
      split_weight_block<4, 12>(mats.m[i], rb);
    return;
  }
  split_row_block<KPW, kLn>(rows, blk - mats.block_end[kSplitMats - 1]);
}

// The same for rows too long for registers: every pass reads them again.
template <bool kLn>
__global__ __launch_bounds__(256) void split_long_rows_kernel(const float* __restrict__ x, int K,
                                                              const float* __restrict__ g,
                                                              const float* __restrict__ b, f16* __restrict__ dst,
                                                              float* __restrict__ inv, long long M, int ksteps) {
  __shared__ float buf[3][4][32];
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const long long rb = blockIdx.x, m = rb * 32 + n;
  const bool valid = m < M;
  const float* row = x + (size_t)(valid ? m : 0) * K;
  float mean = 0.f, rstd = 1.f;
  if (kLn) {
    float s = 0.f;
    for (int ks = wave; ks < ksteps; ks += 4)
      for (int t = 0; t < 8; ++t) {
        const int k = ks * 16 + 8 * h + t;
        s += k < K ? row[k] : 0.f;
      }
    mean = rows_sum(s, buf[0], wave, lane) / (float)K;
    float ss = 0.f;
    for (int ks = wave; ks < ksteps; ks += 4)
      for (int t = 0; t < 8; ++t) {
        const int k = ks * 16 + 8 * h + t;
        const float d = k < K ? row[k] - mean : 0.f;
        ss += d * d;
      }
    rstd = 1.0f / sqrtf(rows_sum(ss, buf[1], wave, lane) / (float)K + 1e-5f);
  }
  auto value = [&](int k) {
    if (k >= K || !valid) return 0.f;
    return kLn ? (row[k] - mean) * rstd * g[k] + (b ? b[k] : 0.f) : row[k];
  };
  float amax = 0.f;
  for (int ks = wave; ks < ksteps; ks += 4)
    for (int t = 0; t < 8; ++t) amax = fmaxf(amax, fabsf(value(ks * 16 + 8 * h + t)));
  amax = rows_max(amax, buf[2], wave, lane);
  const float s = split_scale(amax);
  if (wave == 0 && lane < 32 && valid) inv[m] = split_inv(s);
  for (int ks = wave; ks < ksteps; ks += 4) {
    f16x8 hi, lo;
    for (int t = 0; t < 8; ++t) {
      f16 a, c;
      split_value(value(ks * 16 + 8 * h + t), s, a, c);
      hi[t] = a;
      lo[t] = c;
    }
    f16* d = dst + ((size_t)rb * ksteps + ks) * kFrag;
    *reinterpret_cast<f16x8*>(d + lane * 8) = hi;
    *reinterpret_cast<f16x8*>(d + kFragHalf + lane * 8) = lo;
  }
}

// ---------------------------------------------------------------------------
// Epilogues: four consecutive channels c .. c + 3 of row m (already unscaled).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + __expf(-x)); }

constexpr bool stores_rows(int epi) { return epi == kSplitStore || epi == kSplitHidden; }

// What is added to channels c0 .. c0 + 15 of row m: the residual (stores_rows), the q bias (kSplitQkvg).
template <int kEpi>
__device__ __forceinline__ void load_addend(const SplitGemmEpi& e, long long m, int c0, f32x4 (&r)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (stores_rows(kEpi) && e.res)
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = *reinterpret_cast<const f32x4*>(e.res + (size_t)m * e.ldo + c0 + 4 * q);
  if (kEpi == kSplitQkvg && e.bias && c0 < e.ldo)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int t = 0; t < 4; ++t) r[q][t] = e.bias[c0 + 4 * q + t];
}

template <int kEpi>
__device__ __forceinline__ void epi_quad(const SplitGemmEpi& e, long long m, int c, f32x4 v, f32x4 r) {
  if (stores_rows(kEpi)) {
    float* d = e.out + (size_t)m * e.ldo + c;
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] += r[t];
    *reinterpret_cast<f32x4*>(d) = v;
  } else if (kEpi == kSplitQkvg) {
    // columns [q | k | v | g], c_s each; a quad lies in one part
    const int cs = e.ldo, part = c / cs, cc = c - part * cs;
    if (part == 2 && e.T) {   // v transposed per sequence of T rows, keys contiguous
      const long long sq = m / e.T, t = m - sq * e.T;
      float* col = e.v + ((size_t)sq * cs + cc) * e.T + t;
#pragma unroll
      for (int u = 0; u < 4; ++u) col[(size_t)u * e.T] = v[u];
      return;
    }
    if (part == 0 && e.bias) {
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] += r[t];
    }
    if (part == 3) {
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = sigmoid_f32(v[t]);
    }
    float* d = (part == 0 ? e.out : part == 1 ? e.k : part == 2 ? e.v : e.g) + (size_t)m * cs + cc;
    *reinterpret_cast<f32x4*>(d) = v;
  }
}

// silu(a) b of four hidden channels; amax: the largest magnitude so far.
__device__ __forceinline__ f32x4 swiglu_quad(f32x4 a, f32x4 b, float& amax) {
  f32x4 v;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    v[t] = a[t] * sigmoid_f32(a[t]) * b[t];
    amax = fmaxf(amax, fabsf(v[t]));
  }
  return v;
}

// Hidden channels c .. c + 3 of row m, written as the next product's operand fragments with scale s.
__device__ __forceinline__ void epi_hidden_quad(const SplitGemmEpi& e, long long m, int c, f32x4 v, float s) {
  f16x4 hi, lo;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f16 x, y;
    split_value(split_finite(v[t]), s, x, y);
    hi[t] = x;
    lo[t] = y;
  }
  f16* d = e.hfrag + ((size_t)(m >> 5) * e.hsteps + (c >> 4)) * kFrag +
           (((c >> 3) & 1) * 32 + (int)(m & 31)) * 8 + (c & 4);
  *reinterpret_cast<f16x4*>(d) = hi;
  *reinterpret_cast<f16x4*>(d + kFragHalf) = lo;
}

constexpr int kStageKs = 2;                                   // k-steps per stage
constexpr int kTileStage = 8 * kStageKs * kFrag;              // f16: 4 row blocks of A | 4 of W
constexpr int kTileSmem = 2 * kTileStage * (int)sizeof(f16);  // 64 KB: two workgroups per CU

template <int kEpi>
__global__ __launch_bounds__(256, 2) void split_gemm_kernel(const f16* __restrict__ A, const float* __restrict__ ainv,
                                                            const f16* __restrict__ W, const float* __restrict__ winv,
                                                            SplitGemmEpi e, long long M, int mblocks, int nblocks,
                                                            int ksteps) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f16* smem = reinterpret_cast<f16*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  // XCD-aware order: an XCD takes consecutive tiles, the column tiles of a row tile next to each other, so that
  // a row tile's fragments come from its L2 once.
  const int ncols = (nblocks + 3) / 4, total = (mblocks + 3) / 4 * ncols;
  const int per_xcd = (total + 7) / 8;
  const int item = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (item >= total || (int)(blockIdx.x / 8) >= per_xcd) return;   // uniform over the workgroup
  const int mt = item / ncols, nt = item % ncols;
  const unsigned blk = (unsigned)ksteps * kFrag * 2;   // bytes of one row block
  const __amdgpu_buffer_rsrc_t ra =
      buffer_rsrc(A + (size_t)mt * 4 * ksteps * kFrag, min(mblocks - mt * 4, 4) * blk);
  const __amdgpu_buffer_rsrc_t rw =
      buffer_rsrc(W + (size_t)nt * 4 * ksteps * kFrag, min(nblocks - nt * 4, 4) * blk);
  // copy j (0 .. 15) of an operand: row block j / 4, KB j % 4 of its two k-steps; wave w takes block w
  const unsigned vo = (unsigned)wave * blk + lane * 16;
  auto stage = [&](int ks0) {
    f16* st = smem + ((ks0 / kStageKs) & 1) * kTileStage;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      copy1k_to_lds(ra, st + (wave * 4 + p) * kFragHalf, vo, (unsigned)(ks0 * kFrag * 2 + p * 1024));
      copy1k_to_lds(rw, st + (16 + wave * 4 + p) * kFragHalf, vo, (unsigned)(ks0 * kFrag * 2 + p * 1024));
    }
  };
  f32x16 acc[2][2];   // [column block][row block]
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[j][i] = zero16();
  // kSplitHidden: a stage is the 32 columns of one scale, and its products are added under it.  The next stage's scales
  // are requested ahead of its copies (loads return in order).
  static_assert(kStageKs == 2, "a stage is 32 columns");
  float sc[2], scn[2] = {0.f, 0.f};
  auto load_scales = [&](int ks0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const long long m = ((long long)mt * 4 + wm * 2 + i) * 32 + n;
      scn[i] = ainv[(size_t)(ks0 / 2) * M + (m < M ? m : M - 1)];
    }
  };
  f32x16 part[2][2];   // [column block][row block]: a stage's products, not yet added
  float scp[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i) part[1][i] = zero16();
  auto add_part = [&](int j, const float (&s)[2], int q) {   // a quarter of column block j's
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[j][q >> 1][8 * (q & 1) + t] += part[j][q >> 1][8 * (q & 1) + t] * s[q >> 1];
  };
  if (kEpi == kSplitHidden) load_scales(0);
  stage(0);
#pragma unroll 1
  for (int ks0 = 0; ks0 < ksteps; ks0 += kStageKs) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of the stage landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
#pragma unroll
    for (int i = 0; i < 2; ++i) sc[i] = scn[i];
    if (ks0 + kStageKs < ksteps) {
      if (kEpi == kSplitHidden) load_scales(ks0 + kStageKs);
      stage(ks0 + kStageKs);
    }
    const f16* sa = smem + ((ks0 / kStageKs) & 1) * kTileStage;
    const f16* sw = sa + 4 * kStageKs * kFrag;
    SplitFrag fa[kStageKs][2], fw[kStageKs][2];
#pragma unroll
    for (int ks = 0; ks < kStageKs; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[ks][i] = load_frag(sa + ((wm * 2 + i) * kStageKs + ks) * kFrag, lane);
        fw[ks][i] = load_frag(sw + ((wn * 2 + i) * kStageKs + ks) * kFrag, lane);
      }
    __builtin_amdgcn_sched_barrier(0);
    if (kEpi == kSplitHidden) {
      // a column block's sums (the other's of the stage before, this one's) between the other's products
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 p0 = zero16(), p1 = zero16();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          mfma_split(fw[q & 1][j], fa[q & 1][q >> 1], q < 2 ? p0 : p1);
          add_part(1 - j, j ? sc : scp, q);
          __builtin_amdgcn_sched_barrier(0);
        }
        part[j][0] = p0;
        part[j][1] = p1;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) scp[i] = sc[i];
    } else {
#pragma unroll
      for (int ks = 0; ks < kStageKs; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) mfma_split(fw[ks][j], fa[ks][i], acc[j][i]);
    }
  }
  if (kEpi == kSplitHidden)
#pragma unroll
    for (int q = 0; q < 4; ++q) add_part(1, scp, q);
  const int cb0 = nt * 4 + wn * 2;
  if (cb0 >= nblocks) return;
  // the weight rows' scales, read before the first store
  f32x4 w[2][4];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      w[j][q] = *reinterpret_cast<const f32x4*>(winv + min(cb0 + j, nblocks - 1) * 32 + 16 * h + 4 * q);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const long long m = ((long long)mt * 4 + wm * 2 + i) * 32 + n;
    if (m >= M) continue;   // both lanes of a row
    const float s = kEpi == kSplitHidden ? 1.0f : ainv[m];
    if (kEpi == kSplitSwiGLU) {
      f32x4 v[4];
      float amax = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 a, b;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          a[t] = acc[0][i][4 * q + t] * s * w[0][q][t];
          b[t] = acc[1][i][4 * q + t] * s * w[1][q][t];
        }
        v[q] = swiglu_quad(a, b, amax);
      }
      const float hs = split_scale(fmaxf(amax, __shfl_xor(amax, 32)));
      if (h == 0) e.hinv[(size_t)(cb0 / 2) * M + m] = split_inv(hs);
#pragma unroll
      for (int q = 0; q < 4; ++q) epi_hidden_quad(e, m, cb0 * 16 + 16 * h + 4 * q, v[q], hs);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (cb0 + j >= nblocks) break;
        const int c0 = (cb0 + j) * 32 + 16 * h;
        f32x4 res[4];   // read ahead of the stores (out may be res)
        load_addend<kEpi>(e, m, c0, res);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 v;
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = acc[j][i][4 * q + t] * s * w[j][q][t];
          epi_quad<kEpi>(e, m, c0 + 4 * q, v, res[q]);
        }
      }
    }
  }
}

// One 32-row block x 2 column blocks per workgroup; wave w multiplies the k-steps
// [w, w + 1) * ksteps / 4 straight from memory, the partial sums meet in LDS and
// wave w finishes channels 16 h + 4 w .. + 3 of both column blocks.
template <int kEpi>
__global__ __launch_bounds__(256) void split_gemm_small_kernel(const f16* __restrict__ A,
                                                               const float* __restrict__ ainv,
                                                               const f16* __restrict__ W,
                                                               const float* __restrict__ winv, SplitGemmEpi e,
                                                               long long M, int nblocks, int ksteps) {
  __shared__ __attribute__((aligned(16))) f32x4 part[4][2][4][64];   // [wave][column block][quad][lane]: 32 KB
  __shared__ float hmax[kEpi == kSplitSwiGLU ? 4 : 1][32];
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int ncols = (nblocks + 1) / 2;
  const long long mb = blockIdx.x / ncols;
  const int cb0 = (int)(blockIdx.x % ncols) * 2;
  const bool two = cb0 + 1 < nblocks;
  const int k0 = wave * ksteps / 4, k1 = (wave + 1) * ksteps / 4;
  const f16* pa = A + (size_t)mb * ksteps * kFrag;
  const f16* pw = W + (size_t)cb0 * ksteps * kFrag;
  const f16* pw1 = two ? pw + (size_t)ksteps * kFrag : pw;
  const long long m = mb * 32 + n, mc = m < M ? m : M - 1;
  f32x16 acc[2] = {zero16(), zero16()};
  constexpr int kDepth = 4;   // k-steps requested together
  for (int ks = k0; ks < k1; ks += kDepth) {
    SplitFrag fa[kDepth], f0[kDepth], f1[kDepth];
    float sc[kDepth];
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      const int k = min(ks + d, k1 - 1);
      const size_t o = (size_t)k * kFrag;
      if (kEpi == kSplitHidden) sc[d] = ainv[(size_t)(k / 2) * M + mc];
      fa[d] = load_frag(pa + o, lane);
      f0[d] = load_frag(pw + o, lane);
      f1[d] = load_frag(pw1 + o, lane);
    }
#pragma unroll
    for (int d = 0; d < kDepth; ++d)
      if (ks + d < k1) {
        if (kEpi == kSplitHidden) {
          f32x16 p0 = zero16(), p1 = zero16();
          mfma_split(f0[d], fa[d], p0);
          mfma_split(f1[d], fa[d], p1);
#pragma unroll
          for (int u = 0; u < 16; ++u) {
            acc[0][u] += p0[u] * sc[d];
            acc[1][u] += p1[u] * sc[d];
          }
        } else {
          mfma_split(f0[d], fa[d], acc[0]);
          mfma_split(f1[d], fa[d], acc[1]);
        }
      }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v;
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = acc[j][4 * q + t];
      part[wave][j][q][lane] = v;
    }
  __syncthreads();
  f32x4 sum[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    sum[j] = part[0][j][wave][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const f32x4 v = part[w][j][wave][lane];
#pragma unroll
      for (int t = 0; t < 4; ++t) sum[j][t] += v[t];
    }
  }
  const int c = 16 * h + 4 * wave;
  const float s = kEpi == kSplitHidden ? 1.0f : ainv[mc];
  const f32x4 w0 = *reinterpret_cast<const f32x4*>(winv + cb0 * 32 + c);
  const f32x4 w1 = *reinterpret_cast<const f32x4*>(winv + (cb0 + two) * 32 + c);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    sum[0][t] *= s * w0[t];
    sum[1][t] *= s * w1[t];
  }
  if (kEpi == kSplitSwiGLU) {
    float amax = 0.f;
    const f32x4 v = swiglu_quad(sum[0], sum[1], amax);
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    if (lane < 32) hmax[wave][lane] = amax;
    __syncthreads();
    if (m >= M) return;
    const float hs = split_scale(fmaxf(fmaxf(hmax[0][n], hmax[1][n]), fmaxf(hmax[2][n], hmax[3][n])));
    if (h == 0 && wave == 0) e.hinv[(size_t)(cb0 / 2) * M + m] = split_inv(hs);
    epi_hidden_quad(e, m, cb0 * 16 + c, v, hs);
  } else {
    if (m >= M) return;
    f32x4 r0 = {0.f, 0.f, 0.f, 0.f}, r1 = r0;
    const int c0 = cb0 * 32 + c;
    if (stores_rows(kEpi) && e.res) {
      const float* r = e.res + (size_t)m * e.ldo + c0;
      r0 = *reinterpret_cast<const f32x4*>(r);
      if (two) r1 = *reinterpret_cast<const f32x4*>(r + 32);
    }
    if (kEpi == kSplitQkvg && e.bias) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (c0 < e.ldo) r0[t] = e.bias[c0 + t];
        if (two && c0 + 32 < e.ldo) r1[t] = e.bias[c0 + 32 + t];
      }
    }
    epi_quad<kEpi>(e, m, cb0 * 32 + c, sum[0], r0);
    if (two) epi_quad<kEpi>(e, m, (cb0 + 1) * 32 + c, sum[1], r1);
  }
}

// Rows of 128 channels, held as operand fragments by the wave that reads them (kLn: normalised, the affine folded
// into W and wbias): 4 waves x 32 rows, the weights walked in blocks of 32 output channels (16 KB of fragments)
// through double-buffered LDS, `per` of them by a workgroup.  For K = 128 this replaces the separate fragment pass
// and the short k-loop of the tiled kernel.
constexpr int kR128Block = 8 * kFrag;   // f16 elements of one 32-channel block
constexpr int kR128MaxN = 512;          // output channels

template <int kEpi, bool kLn>
__global__ __launch_bounds__(256, 3) void split_gemm_r128_kernel(const float* __restrict__ x, const f16* __restrict__ W,
                                                                 const float* __restrict__ winv,
                                                                 const float* __restrict__ wbias, SplitGemmEpi e,
                                                                 long long M, int nblocks, int per) {
  __shared__ __attribute__((aligned(16))) f16 smem[2][kR128Block];
  __shared__ __attribute__((aligned(16))) float swinv[kR128MaxN], sbias[kLn ? kR128MaxN : 4];
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(W, (unsigned)nblocks * kR128Block * 2);
  auto stage = [&](int cb) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = wave * 4 + q;
      copy1k_to_lds(rw, &smem[cb & 1][c * kFragHalf], lane * 16, (unsigned)(cb * kR128Block * 2 + c * 1024));
    }
  };
  const int first = blockIdx.y * per, last = min(first + per, nblocks);   // first < nblocks
  stage(first);
  stage_floats(swinv, winv, nblocks * 32, nblocks * 32, kLn ? 1.0f / kNormScale : 1.0f);
  if (kLn) stage_floats(sbias, wbias, nblocks * 32, nblocks * 32);
  const long long m = ((long long)blockIdx.x * 4 + wave) * 32 + n;
  const bool valid = m < M;
  SplitFrag xf[8];
  float xinv;   // kLn: besides 1 / kNormScale, in swinv
  {
    float v[64];
    load_row_half<128>(x + (size_t)(valid ? m : 0) * 128, h, v);
    xinv = kLn ? normalized_row_half<128>(v, xf) : split_row_half<128>(v, xf);
  }
#pragma unroll 1
  for (int cb = first; cb < last; ++cb) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of block cb landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
    if (cb + 1 < last) stage(cb + 1);
    f32x16 acc = zero16();
    mfma_block<8>(smem[cb & 1], xf, lane, acc);
    if (kLn) undo_gain(acc, xinv);
    if (valid) {
      const int c0 = cb * 32 + 16 * h;
      f32x4 res[4];
      load_addend<kEpi>(e, m, c0, res);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (kLn) v = *reinterpret_cast<const f32x4*>(&sbias[c0 + 4 * q]);
        const f32x4 w = *reinterpret_cast<const f32x4*>(&swinv[c0 + 4 * q]);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] += (kLn ? acc[4 * q + t] : acc[4 * q + t] * xinv) * w[t];
        epi_quad<kEpi>(e, m, c0 + 4 * q, v, res[q]);
      }
    }
  }
}

}  // namespace

int split_gemm_r128(int epi, const float* x, const f16* W, const float* winv, const float* wbias,
                    const SplitGemmEpi& e, long long M, int N, hipStream_t stream, const char* name) {
  // As many parts of the columns as fill three workgroups per CU (its resident number): the parts read the same rows,
  // from L2, and compute the same bits.  Atom attention (us, with one part / this many): 384 rows 66 / 32, 6144 rows
  // 75 / 47, 12288 rows 91 / 68, 23040 rows 101 / 87, 49152 rows 151 / 140; one workgroup per CU: 32, 49, 74, 101, 151.
  const long long wgs = (M + 127) / 128, nblocks = N / 32, resident = 3LL * compute_units();
  const long long parts = std::min(nblocks, std::max(1LL, resident / wgs)), per = (nblocks + parts - 1) / parts;
  const dim3 grid((unsigned)wgs, (unsigned)((nblocks + per - 1) / per));
  if (N > kR128MaxN) return set_error(BIOEMU_ERR_UNSUPPORTED, "%s: %d output channels", name, N);
  KernelTimerScope timed(name, stream);
#define BIOEMU_R128(E, L)                                                                                        \
  hipLaunchKernelGGL((split_gemm_r128_kernel<E, L>), grid, dim3(256), 0, stream, x, W, winv, wbias, e, M, N / 32, \
                     (int)per)
  if (epi == kSplitStore && !wbias)
    BIOEMU_R128(kSplitStore, false);
  else if (epi == kSplitQkvg && !wbias)
    BIOEMU_R128(kSplitQkvg, false);
  else if (epi == kSplitQkvg)
    BIOEMU_R128(kSplitQkvg, true);
  else
    return set_error(BIOEMU_ERR_UNSUPPORTED, "%s: epilogue %d", name, epi);
#undef BIOEMU_R128
  return check_launch(name);
}

int split_weights(const SplitMats& mats, int count, hipStream_t stream) {
  int blocks = 0;
  for (int i = 0; i < count; ++i) blocks = std::max(blocks, (mats.m[i].rows + 31) / 32);
  // the memory to clear: 64 KB a workgroup, beside the weights
  if (mats.zero_bytes) blocks = std::max(blocks, (int)std::min<size_t>((mats.zero_bytes + 65535) / 65536, 2048));
  KernelTimerScope timed("f32_split_weights", stream);
  const dim3 grid(blocks, count + (mats.zero_bytes ? 1 : 0));
  hipLaunchKernelGGL(split_weights_kernel, grid, dim3(64 * kSwWaves), 0, stream, mats, count);
  return check_launch("f32_split_weights");
}

int split_prep(SplitMats mats, int count, SplitRows r, hipStream_t stream) {
  const long long rblocks = (r.M + 31) / 32;
  r.ksteps = split_ksteps(r.K);
  const bool is_long = r.K > kSplitMaxK;
  if (count && is_long) {
    const int rc = split_weights(mats, count, stream);
    if (rc) return rc;
    count = 0;
  }
  int wblocks = 0;
  for (int i = 0; i < kSplitMats; ++i) {
    if (i < count) wblocks += (mats.m[i].rows + 31) / 32;
    mats.block_end[i] = wblocks;
  }
  const int kpw = (r.ksteps + 3) / 4;
  const dim3 grid((unsigned)(wblocks + rblocks)), block(256);
  KernelTimerScope timed("f32_split_rows", stream);
  if (is_long) {
    if (r.g)
      hipLaunchKernelGGL(split_long_rows_kernel<true>, grid, block, 0, stream, r.x, r.K, r.g, r.b, r.dst, r.inv,
                         r.M, r.ksteps);
    else
      hipLaunchKernelGGL(split_long_rows_kernel<false>, grid, block, 0, stream, r.x, r.K, r.g, r.b, r.dst, r.inv,
                         r.M, r.ksteps);
    return check_launch("f32_split_rows");
  }
#define BIOEMU_SPLIT_PREP(KPW)                                                                  \
  do {                                                                                          \
    if (r.g)                                                                                    \
      hipLaunchKernelGGL((split_prep_kernel<KPW, true>), grid, block, 0, stream, mats, r);      \
    else                                                                                        \
      hipLaunchKernelGGL((split_prep_kernel<KPW, false>), grid, block, 0, stream, mats, r);     \
  } while (0)
  if (kpw <= 2)
    BIOEMU_SPLIT_PREP(2);
  else if (kpw <= 6)
    BIOEMU_SPLIT_PREP(6);
  else
    BIOEMU_SPLIT_PREP(12);
#undef BIOEMU_SPLIT_PREP
  return check_launch("f32_split_rows");
}

int split_gemm(int epi, const f16* A, const float* ainv, const f16* W, const float* winv, const SplitGemmEpi& e,
               long long M, int K, int N, hipStream_t stream, const char* name) {
  const int mb = (int)((M + 31) / 32), nb = N / 32, ks = split_ksteps(K);
  const long long tiles = (long long)((mb + 3) / 4) * ((nb + 3) / 4);
  const bool small = tiles < kSplitTiledMin;
  KernelTimerScope timed(name, stream);
#define BIOEMU_SPLIT_GEMM(E)                                                                                          \
  do {                                                                                                                \
    if (small)                                                                                                        \
      hipLaunchKernelGGL(split_gemm_small_kernel<E>, dim3((unsigned)(mb * ((nb + 1) / 2))), dim3(256), 0, stream, A, \
                         ainv, W, winv, e, M, nb, ks);                                                                \
    else {                                                                                                            \
      const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void*>(split_gemm_kernel<E>),                  \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, kTileSmem);               \
      if (rc != hipSuccess) return set_error(BIOEMU_ERR_LAUNCH, "%s: %s", name, hipGetErrorString(rc));               \
      hipLaunchKernelGGL(split_gemm_kernel<E>, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), kTileSmem, stream,  \
                         A, ainv, W, winv, e, M, mb, nb, ks);                                                         \
    }                                                                                                                 \
  } while (0)
  switch (epi) {
    case kSplitStore: BIOEMU_SPLIT_GEMM(kSplitStore); break;
    case kSplitSwiGLU: BIOEMU_SPLIT_GEMM(kSplitSwiGLU); break;
    case kSplitHidden: BIOEMU_SPLIT_GEMM(kSplitHidden); break;
    default: BIOEMU_SPLIT_GEMM(kSplitQkvg); break;
  }
#undef BIOEMU_SPLIT_GEMM
  return check_launch(name);
}

}  // namespace bioemu
