// Row transition in fp32 on split f16 operands (split.h): rows of 128 or 64 channels
//   out = (res +) fc3(silu(fc1(xn)) * fc2(xn)),  xn = LN(x) or x
// in one pass over memory (Transition.forward, src/bioemu2/biomoa/ops/transition.py:52-91).
//
// A workgroup is 8 waves x 32 rows.  A wave keeps its rows as operand fragments
// in registers (64 VGPRs at c = 128) with the 32 x c output accumulator; the
// hidden dimension is walked in chunks of 32, whose weights (fc1 and fc2 rows,
// fc3 columns, hi and lo: 48 KB at c = 128) arrive in LDS by copies that write it
// directly, double-buffered.  A hidden value never leaves registers: silu(a) b
// comes out of fc1 / fc2 as lane (row n, half h) = hidden 16 h + u, which is the
// fc3 B operand of k-step j when lane half h supplies hidden 16 h + 8 j + t; the
// fc3 fragments are read with the same permutation.  A row's hidden scale follows
// its largest value so far, with three bits to spare before the next step; a step
// rescales the accumulators (by a power of two).  A LayerNorm's affine is folded into
// fc1 and fc2, so the rows are only centred and divided by their deviation.
//
// Few rows take the separate products of split_gemm.hip instead (the rule and both times: fp32.hip).
//
// Bound by the matrix cores and the gating VALU work of the same waves (two waves per
// SIMD): 590k rows, 128 -> 256, 0.45 ms (259 TFLOP/s of fp32 products, 776 of f16)
// against 2.1 ms for LayerNorm, SwiGLU and output products on fp32 MFMA through
// memory; 111k rows, 128 -> 512: 0.151 ms against 0.67.
#include "split.h"
#include "split_rows.h"

namespace bioemu {
namespace {

constexpr int kWaves = 8;

template <int C>
struct TGeo {
  static constexpr int KS = C / 16;
  static constexpr int W3 = 2 * KS * kFrag;               // f16 offset of the fc3 fragments in a chunk
  static constexpr int Chunk = (2 * KS + C / 16) * kFrag; // f16 elements: fc1 | fc2 | fc3 [C / 32 blocks][2 k-steps]
  static constexpr int Copies = Chunk / kFragHalf;        // 1 KB copies
  static constexpr int Smem = 2 * Chunk * 2;
};

template <int C, bool kLn>
__global__ __launch_bounds__(64 * kWaves, 2) void transition_rows_f32_kernel(
    const float* x, const float* res, const f16* __restrict__ W, const float* __restrict__ inv12,
    const float* __restrict__ bias12, const float* __restrict__ inv3, float* out, long long M, int chunks) {
  using G = TGeo<C>;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f16* smem = reinterpret_cast<f16*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(W, (unsigned)chunks * G::Chunk * 2);
  static_assert(G::Copies % kWaves == 0, "copies split evenly over the waves");
  auto stage = [&](int hc) {
    f16* st = smem + (hc & 1) * G::Chunk;
#pragma unroll
    for (int q = 0; q < G::Copies / kWaves; ++q) {
      const int c = wave + kWaves * q;
      copy1k_to_lds(rw, st + c * kFragHalf, lane * 16, (unsigned)(hc * G::Chunk * 2 + c * 1024));
    }
  };
  stage(0);
  // 1 / scale of the fc1 and fc2 rows of every chunk, [chunk][fc1 | fc2][32], and of the fc3 rows; the biases (W beta)
  // of fc1 and fc2
  float* sinv = reinterpret_cast<float*>(smem_raw + 2 * G::Chunk * 2);
  float *sinv3 = sinv + chunks * 64, *sbias = sinv3 + C;
  stage_floats(sinv, inv12, chunks * 64, chunks * 64, kLn ? 1.0f / kNormScale : 1.0f);
  stage_floats(sinv3, inv3, C, C);
  if (kLn)
    for (int i = threadIdx.x; i < chunks * 64; i += 64 * kWaves)
      sbias[i] = bias12[(i & 32 ? chunks * 32 : 0) + (i >> 6) * 32 + (i & 31)];
  const long long m = ((long long)blockIdx.x * kWaves + wave) * 32 + n;
  const bool valid = m < M;
  SplitFrag xf[G::KS];
  float xinv;   // kLn: besides 1 / kNormScale, in sinv
  {
    float v[C / 2];
    load_row_half<C>(x + (size_t)(valid ? m : 0) * C, h, v);
    xinv = kLn ? normalized_row_half<C>(v, xf) : split_row_half<C>(v, xf);
  }
  float hs = split_scale(0.f);   // the row's hidden scale
  f32x16 acc[C / 32];
#pragma unroll
  for (int cb = 0; cb < C / 32; ++cb) acc[cb] = zero16();
#pragma unroll 1
  for (int hc = 0; hc < chunks; ++hc) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of chunk hc landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
    if (hc + 1 < chunks) stage(hc + 1);
    const f16* st = smem + (hc & 1) * G::Chunk;
    f32x16 a = zero16(), gt = zero16();
    mfma_block2<G::KS>(st, st + G::KS * kFrag, xf, xf, lane, a, gt);
    if (kLn) {
      undo_gain(a, xinv);
      undo_gain(gt, xinv);
    }
    SplitFrag hf[2];
    const float *sb = sbias + hc * 64 + 16 * h, *si = sinv + hc * 64 + 16 * h;
    float hv[16], amax = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float p = kLn ? a[u] * si[u] + sb[u] : a[u] * xinv * si[u];
      const float q = kLn ? gt[u] * si[32 + u] + sb[32 + u] : gt[u] * xinv * si[32 + u];
      hv[u] = p * sigmoidf_fast(p) * q;
      amax = fmaxf(amax, fabsf(hv[u]));
    }
    amax = max_halves(amax);
    if (__any(amax * hs >= 32768.f)) {   // each row for itself
      const float ns = amax * hs >= 32768.f ? split_scale(amax) * 0.125f : hs, ratio = ns * split_inv(hs);
#pragma unroll
      for (int cb = 0; cb < C / 32; ++cb)
#pragma unroll
        for (int u = 0; u < 16; ++u) acc[cb][u] *= ratio;
#pragma unroll
      for (int u = 0; u < 16; ++u) hv[u] = split_finite(hv[u]);
      hs = ns;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      f16 hi, lo;
      split_value(hv[u], hs, hi, lo);
      hf[u >> 3].hi[u & 7] = hi;
      hf[u >> 3].lo[u & 7] = lo;
    }
#pragma unroll
    for (int cb = 0; cb < C / 32; ++cb)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        // lane (n, h) takes columns 16 h + 8 j + t: half j of k-step h
        mfma_split(load_frag(st + G::W3 + (2 * cb + h) * kFrag, j * 32 + n), hf[j], acc[cb]);
  }
  if (!valid) return;
  const float hinv = split_inv(hs);
#pragma unroll
  for (int cb = 0; cb < C / 32; ++cb) {
    const size_t off = (size_t)m * C + cb * 32 + 16 * h;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 o;
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] = acc[cb][4 * q + t] * hinv * sinv3[cb * 32 + 16 * h + 4 * q + t];
      if (res) {
        const f32x4 r = *reinterpret_cast<const f32x4*>(res + off + 4 * q);
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] += r[t];
      }
      *reinterpret_cast<f32x4*>(out + off + 4 * q) = o;
    }
  }
}

template <int C, bool kLn>
int launch(const float* x, const float* res, const f16* W, const float* inv12, const float* bias12, const float* inv3,
           float* out, long long M, int hidden, hipStream_t stream, const char* name) {
  const int smem = TGeo<C>::Smem + (4 * hidden + C) * 4;
  const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void*>(transition_rows_f32_kernel<C, kLn>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            TGeo<C>::Smem + (4 * kTransitionMaxHidden + C) * 4);
  if (rc != hipSuccess) return set_error(BIOEMU_ERR_LAUNCH, "%s: %s", name, hipGetErrorString(rc));
  KernelTimerScope timed(name, stream);
  const unsigned grid = (unsigned)((M + 32 * kWaves - 1) / (32 * kWaves));
  hipLaunchKernelGGL((transition_rows_f32_kernel<C, kLn>), dim3(grid), dim3(64 * kWaves), (unsigned)smem, stream, x,
                     res, W, inv12, bias12, inv3, out, M, hidden / 32);
  return check_launch(name);
}

}  // namespace

size_t split_transition_weight_elems(int64_t C, int64_t hidden) {
  return (size_t)(hidden / 32) * (C == 128 ? TGeo<128>::Chunk : TGeo<64>::Chunk);
}

int split_transition_rows(const float* x, const float* res, const float* norm_w, const float* norm_b,
                          const float* fc1, const float* fc2, const float* fc3, f16* W, float* scales, float* out,
                          long long M, int C, int hidden, hipStream_t stream, const char* name) {
  const int KS = C / 16;
  const long long chunk = C == 128 ? TGeo<128>::Chunk : TGeo<64>::Chunk;
  float *inv12 = scales, *inv3 = inv12 + 2 * hidden, *bias12 = inv3 + C;
  SplitMats mats{};
  mats.m[0] = with_fold(SplitMat{fc1, W, inv12, nullptr, hidden, C, KS, KS, chunk, 0, 2, nullptr, nullptr, nullptr},
                        norm_w, norm_b, norm_w ? bias12 : nullptr);
  mats.m[1] = with_fold(SplitMat{fc2, W + (size_t)KS * kFrag, inv12 + 32, nullptr, hidden, C, KS, KS, chunk, 0, 2,
                                 nullptr, nullptr, nullptr},
                        norm_w, norm_b, norm_w ? bias12 + hidden : nullptr);
  mats.m[2] = SplitMat{fc3, W + (size_t)2 * KS * kFrag, inv3, nullptr, C, hidden, hidden / 16, 2, 2 * kFrag, chunk, 1,
                       nullptr, nullptr, nullptr};
  const int rc = split_weights(mats, 3, stream);
  if (rc) return rc;
#define BIOEMU_TRANSITION(CC, LN) \
  return launch<CC, LN>(x, res, W, inv12, bias12, inv3, out, M, hidden, stream, name)
  if (C == 128) {
    if (norm_w) BIOEMU_TRANSITION(128, true);
    BIOEMU_TRANSITION(128, false);
  }
  if (norm_w) BIOEMU_TRANSITION(64, true);
  BIOEMU_TRANSITION(64, false);
#undef BIOEMU_TRANSITION
}

}  // namespace bioemu
