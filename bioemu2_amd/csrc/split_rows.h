// Rows of fp32 activations held in registers as split operands (split.h): the
// two lanes (n, 0) and (n, 1) of row slot n hold alternate 8-channel chunks, lane
// half h channels 16 s + 8 h .. + 7 of every k-step s, i.e. the MFMA operand layout.
#pragma once

#include "split.h"

namespace bioemu {

// This lane's C / 2 channels of a row (16-byte aligned).
template <int C>
__device__ __forceinline__ void load_row_half(const float* row, int h, float (&v)[C / 2]) {
#pragma unroll
  for (int s = 0; s < C / 16; ++s)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(row + 16 * s + 8 * h + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[8 * s + 4 * q + e] = t[e];
    }
}

// Largest magnitude of the row.
template <int C>
__device__ __forceinline__ float row_absmax(const float (&v)[C / 2]) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < C / 2; ++i) amax = fmaxf(amax, fabsf(v[i]));
  return fmaxf(amax, __shfl_xor(amax, 32));
}

// Fragments of v * s, s a power of two.
template <int C>
__device__ __forceinline__ void split_half(const float (&v)[C / 2], float s, SplitFrag* f) {
#pragma unroll
  for (int i = 0; i < C / 2; ++i) {
    f16 hi, lo;
    split_value(v[i], s, hi, lo);
    f[i >> 3].hi[i & 7] = hi;
    f[i >> 3].lo[i & 7] = lo;
    if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);   // a k-step's fp32 values die before the next one's fragments
  }
}

// The row's fragments under its own scale; returns 1 / scale.
template <int C>
__device__ __forceinline__ float split_row_half(const float (&v)[C / 2], SplitFrag (&f)[C / 16]) {
  const float s = split_scale(row_absmax<C>(v));
  split_half<C>(v, s, f);
  return split_inv(s);
}

// A normalised row of up to 256 channels is below 16 in magnitude: it takes this scale, which brings it below 2^14.
// Rows whose deviation is far below the LayerNorm's epsilon come out small, and take this scale times norm_gain.
constexpr float kNormScale = 1024.f;

// 2^k for a normalised row of mean square t (the variance over variance plus epsilon): 1 down to t = 2^-8, below it
// what brings the root mean square into [0.7, 1.42).  With 22.6 times that (256 channels) the largest magnitude stays
// below 2^14.6.  Exact split_inv of it.
__device__ __forceinline__ float norm_gain(float t) {
  const int e = 127 - (int)((__builtin_bit_cast(uint32_t, t) >> 23) & 0xffu);   // 2^-e <= t
  return __builtin_bit_cast(float, (uint32_t)(127 + (e > 8 ? e >> 1 : 0)) << 23);
}

// Sum of the row halves' values f(0) .. f(C / 2 - 1) over lanes l and l ^ 32.  Eight partial sums: a channel close to
// its row's mean under a large weight shows the mean's rounding, which one chain of C / 2 additions would double.
template <int C, typename F>
__device__ __forceinline__ float row_sum(F f) {
  float p[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = f(i);
#pragma unroll
  for (int i = 8; i < C / 2; ++i) p[i & 7] += f(i);
#pragma unroll
  for (int off = 4; off >= 1; off >>= 1)
#pragma unroll
    for (int i = 0; i < off; ++i) p[i] += p[i + off];
  return p[0] + __shfl_xor(p[0], 32);
}

// Centres the row (v -= mean) and returns rstd = 1 / sqrt(biased variance + 1e-5): the affine-free LayerNorm in fp32,
// two passes, over the C channels of lanes l and l ^ 32; and the row's norm_gain.
template <int C>
__device__ __forceinline__ float center_row_half(float (&v)[C / 2], float& gain) {
  const float mean = row_sum<C>([&](int i) { return v[i]; }) * (1.0f / C);
#pragma unroll
  for (int i = 0; i < C / 2; ++i) v[i] -= mean;
  const float var = row_sum<C>([&](int i) { return v[i] * v[i]; }) * (1.0f / C), rstd = 1.0f / sqrtf(var + 1e-5f);
  gain = norm_gain(var * rstd * rstd);
  return rstd;
}

// Fragments of kNormScale * gain * v * rstd.  v * rstd is rounded to fp32 by itself (see split_value).
template <int C>
__device__ __forceinline__ void split_normalized(float (&v)[C / 2], float rstd, float gain, SplitFrag* f) {
#pragma clang fp contract(off)
#pragma unroll
  for (int i = 0; i < C / 2; ++i) v[i] = v[i] * rstd;
  split_half<C>(v, kNormScale * gain, f);
}

// Fragments of the normalised row, times kNormScale * norm_gain; returns 1 / norm_gain.
template <int C>
__device__ __forceinline__ float normalized_row_half(float (&v)[C / 2], SplitFrag (&f)[C / 16]) {
  float gain;
  const float rstd = center_row_half<C>(v, gain);
  split_normalized<C>(v, rstd, gain, f);
  return split_inv(gain);
}

// acc *= xinv, left out where no row of the wave has a gain.
__device__ __forceinline__ void undo_gain(f32x16& acc, float xinv) {
  if (__any(xinv != 1.0f))
#pragma unroll
    for (int u = 0; u < 16; ++u) acc[u] *= xinv;
}

// Copies `kb` KB of fragments into LDS, split over the workgroup's waves.
__device__ __forceinline__ void stage_fragments(const f16* W, f16* smem, int kb, int waves, int wave, int lane) {
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(W, (unsigned)kb * 1024);
  for (int c = wave; c < kb; c += waves) copy1k_to_lds(rw, smem + c * kFragHalf, lane * 16, (unsigned)c * 1024);
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  __syncthreads();
}

// Copies `count` floats times `scale` into LDS (whole workgroup; no barrier).  Epilogues read their biases and scales
// from LDS: a global load there would wait for every store before it (vmcnt counts both, in order).
__device__ __forceinline__ void stage_floats(float* dst, const float* __restrict__ src, int count, int padded,
                                             float scale = 1.0f) {
  for (int i = threadIdx.x; i < padded; i += blockDim.x) dst[i] = i < count ? src[i] * scale : 0.f;
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
// Fused transition over rows of C = 64 or 128 channels (split_transition.hip): hidden % 32 == 0, at most
// kTransitionMaxHidden.  `W` holds split_transition_weight_elems f16, `scales` split_transition_scales floats.
constexpr int kTransitionMaxHidden = 2048;
constexpr int64_t kTransitionFusedRows128 = 18432, kTransitionFusedRows64 = 12288;   // fewest rows worth it
inline size_t split_transition_scales(int64_t C, int64_t hidden) { return (size_t)(4 * hidden + C); }
size_t split_transition_weight_elems(int64_t C, int64_t hidden);
int split_transition_rows(const float* x, const float* res, const float* norm_w, const float* norm_b,
                          const float* fc1, const float* fc2, const float* fc3, f16* W, float* scales, float* out,
                          long long M, int C, int hidden, hipStream_t stream, const char* name);

// out [P][128] = LN([x1 | x2]) W^T of P rows of 128 + 128 channels (split_pair.hip); W, winv, wbias: 128 x 256
// weights with the LayerNorm folded in (SplitMat).
int split_cat_proj(const float* x1, const float* x2, const f16* W, const float* winv, const float* wbias, float* out,
                   long long P, hipStream_t stream, const char* name);

// Pair bias LN(z) W^T of P < 2^31 rows of 128 channels, head-major: row p = (outer, r, c) -> out[outer][head][r][c],
// rows ld apart, times `scale` (split_pair.hip); W, winv, wbias: H x 128 weights with the LayerNorm folded in, H <= 64.
int split_pair_bias(const float* z, const f16* W, const float* winv, const float* wbias, float* out, long long P,
                    int nrows, int ncols, int ld, int H, float scale, hipStream_t stream, const char* name);

// Attention of BM = B * mult sequences of N tokens, heads of 24 or 32 channels (split_attn.hip): q, k, v, g, go
// [BM][N][c_s], bias [B][H][N][ld] times log2(e), mask [B][N] or, mask_per_copy, [BM][N].  Scratch: kv
// split_attn_kv_elems, kvinv 2 floats and words one 32-bit word per 32 keys of every (sequence, head).
struct SplitAttn {
  const float *q, *k, *v, *g, *bias;
  const uint8_t* mask;
  float* go;
  f16* kv;
  float* kvinv;
  uint32_t* words;
  int BM, mult, N, ld, H, c_s, mask_per_copy;
};
size_t split_attn_kv_elems(int64_t BM, int64_t H, int64_t N);
int split_attn(const SplitAttn& a, hipStream_t stream, const char* name);

// Triangle multiplication of 128 channels (split_trimul.hip): the arguments of bioemu_trimul_fwd_f32.
size_t split_trimul_workspace_bytes(int64_t B, int64_t N);
int split_trimul(const float* x, const uint8_t* mask, const float* norm_in_w, const float* norm_in_b,
                 const float* p_in_w, const float* g_in_w, const float* norm_out_w, const float* norm_out_b,
                 const float* p_out_w, const float* g_out_w, float* out, void* workspace, int64_t B, int64_t N,
                 int outgoing, int residual, hipStream_t stream);

}  // namespace bioemu
