// Projections of fp32 pair rows on split f16 operands (split.h), one pass over
// the rows each: a wave normalises 32 rows in registers and multiplies them with
// weights that stay in LDS for the whole launch (grid of resident workgroups,
// waves walking row tiles).  Both are bound by reading the rows: the conditioning
// projection (590k rows of 256, 906 MB) takes 0.214 ms, 4.2 TB/s, against 1.17 ms for
// a LayerNorm pass and an fp32-MFMA product; the 16-head pair bias (590k rows of 128,
// 340 MB) 0.078 ms, 4.4 TB/s (a stream read and written on this card: 6.3), against
// 0.109 ms for one thread per row on the VALU.  Rows requested a tile ahead and biases read from LDS
// (a global load in the epilogue waits for the stores before it) took it from 0.097.
#include <algorithm>

#include "split.h"
#include "split_rows.h"

namespace bioemu {
namespace {

constexpr int kCatWaves = 8;   // with all four column blocks in LDS
constexpr int kCatWeights = 4 * 16 * kFrag;               // f16: [4 column blocks][16 k-steps]
constexpr int kCatScales = 2 * 128 * 4;                   // bytes: the biases and the weights' scales
constexpr int kCatSmem = kCatScales + kCatWeights * (int)sizeof(f16);

__global__ __launch_bounds__(64 * kCatWaves, 2) void cat_proj_f32_kernel(
    const float* __restrict__ x1, const float* __restrict__ x2, const f16* __restrict__ W,
    const float* __restrict__ winv, const float* __restrict__ wbias, float* __restrict__ out, long long P, int tiles,
    int per) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float *sbias = reinterpret_cast<float*>(smem_raw), *swinv = sbias + 128;
  f16* smem = reinterpret_cast<f16*>(swinv + 128);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int waves = blockDim.x / 64, cb0 = blockIdx.y * per;   // column blocks cb0 .. cb0 + per - 1
  stage_floats(sbias, wbias + cb0 * 32, per * 32, per * 32);
  stage_floats(swinv, winv + cb0 * 32, per * 32, per * 32, 1.0f / kNormScale);
  stage_fragments(W + cb0 * 16 * kFrag, smem, per * 32, waves, wave, lane);
  // half of the next tile's rows is requested as soon as this tile's are fragments, ahead of its products and stores
  float a[64];
  auto row_of = [&](int tile) { return (size_t)std::min((long long)tile * 32 + n, P - 1) * 128; };
  const int first = blockIdx.x * waves + wave, step = gridDim.x * waves;
  if (first < tiles) load_row_half<128>(x1 + row_of(first), h, a);
#pragma unroll 1
  for (int tile = first; tile < tiles; tile += step) {
    const long long m = (long long)tile * 32 + n;
    const bool valid = m < P;
    SplitFrag xf[16];
    float xinv;
    {
      float c[64];
      load_row_half<128>(x2 + row_of(tile), h, c);
      // LayerNorm statistics over the concatenation
      const float mean = row_sum<128>([&](int i) { return a[i] + c[i]; }) * (1.0f / 256.0f);
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        a[i] -= mean;
        c[i] -= mean;
      }
      const float var = row_sum<128>([&](int i) { return a[i] * a[i] + c[i] * c[i]; }) * (1.0f / 256.0f);
      const float rstd = 1.0f / sqrtf(var + 1e-5f), gain = norm_gain(var * rstd * rstd);
      split_normalized<128>(a, rstd, gain, xf);
      split_normalized<128>(c, rstd, gain, xf + 8);
      xinv = split_inv(gain);
    }
    if (tile + step < tiles) load_row_half<128>(x1 + row_of(tile + step), h, a);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int cb = 0; cb < per; ++cb) {
      const f16* w = smem + cb * 16 * kFrag;
      f32x16 acc = zero16();
      mfma_block<16>(w, xf, lane, acc);
      undo_gain(acc, xinv);
      if (valid) {
        const int c0 = cb * 32 + 16 * h;
        float* d = out + (size_t)m * 128 + cb0 * 32 + c0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 v = *reinterpret_cast<const f32x4*>(sbias + c0 + 4 * q);
          const f32x4 wi = *reinterpret_cast<const f32x4*>(swinv + c0 + 4 * q);
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] += acc[4 * q + t] * wi[t];
          *reinterpret_cast<f32x4*>(d + 4 * q) = v;
        }
      }
    }
  }
}

// Heads are the MFMA rows, pair rows its columns: register u of lane (n, h) is
// head 32 hb + 16 h + u of pair n, so a store writes 32 consecutive columns.
__global__ __launch_bounds__(256, 2) void pair_bias_split_kernel(const float* __restrict__ z, const f16* __restrict__ W,
                                                                 const float* __restrict__ winv,
                                                                 const float* __restrict__ wbias,
                                                                 float* __restrict__ out, unsigned P, unsigned nrows,
                                                                 unsigned ncols, int ld, int H, float scale, int tiles) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f16* smem = reinterpret_cast<f16*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int nhb = (H + 31) / 32;
  float* sbias = reinterpret_cast<float*>(smem + nhb * 8 * kFrag);
  float* swinv = sbias + nhb * 32;
  stage_floats(sbias, wbias, H, nhb * 32);
  stage_floats(swinv, winv, nhb * 32, nhb * 32, 1.0f / kNormScale);
  stage_fragments(W, smem, nhb * 16, 4, wave, lane);
  float v[64];
  auto load_rows = [&](int tile) { load_row_half<128>(z + (size_t)min((unsigned)tile * 32 + n, P - 1) * 128, h, v); };
  const int first = blockIdx.x * 4 + wave, step = gridDim.x * 4;
  if (first < tiles) load_rows(first);
#pragma unroll 1
  for (int tile = first; tile < tiles; tile += step) {
    const unsigned p = (unsigned)tile * 32 + n;
    const bool valid = p < P;
    SplitFrag xf[8];
    const float xinv = normalized_row_half<128>(v, xf);
    if (tile + step < tiles) load_rows(tile + step);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned rr = p / ncols, col = p - rr * ncols, outer = rr / nrows, r = rr - outer * nrows;
#pragma unroll 1
    for (int hb = 0; hb < nhb; ++hb) {
      f32x16 acc = zero16();
      mfma_block<8>(smem + hb * 8 * kFrag, xf, lane, acc);
      undo_gain(acc, xinv);
      const int h0 = hb * 32 + 16 * h;
      if (valid) {
        float* d = out + (((size_t)outer * H + h0) * nrows + r) * ld + col;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          if (h0 + u < H) *d = (acc[u] * swinv[h0 + u] + sbias[h0 + u]) * scale;
          d += (size_t)nrows * ld;
        }
      }
    }
  }
}

}  // namespace

int split_cat_proj(const float* x1, const float* x2, const f16* W, const float* winv, const float* wbias, float* out,
                   long long P, hipStream_t stream, const char* name) {
  const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void*>(cat_proj_f32_kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, kCatSmem);
  if (rc != hipSuccess) return set_error(BIOEMU_ERR_LAUNCH, "%s: %s", name, hipGetErrorString(rc));
  const int tiles = (int)((P + 31) / 32);
  // Few tiles: a column block (and 32 KB of weights) a workgroup, four waves of which two workgroups share a CU, as
  // long as that is one round of workgroups.  us of the projection and two transitions, all columns / this: 1600 rows
  // 53 / 46, 8100 rows 78 / 71, 16384 rows 91 / 88; past one round, 32400 rows 110 / 123.  The same bits.
  const int cus = compute_units();
  const bool few = tiles <= 2 * cus;
  const int waves = few ? 4 : kCatWaves, per = few ? 1 : 4;
  const int grid = std::min((tiles + waves - 1) / waves, cus);
  KernelTimerScope timed(name, stream);
  hipLaunchKernelGGL(cat_proj_f32_kernel, dim3((unsigned)grid, 4 / per), dim3(64 * waves),
                     kCatScales + per * 16 * kFrag * (int)sizeof(f16), stream, x1, x2, W, winv, wbias, out, P, tiles,
                     per);
  return check_launch(name);
}

int split_pair_bias(const float* z, const f16* W, const float* winv, const float* wbias, float* out, long long P,
                    int nrows, int ncols, int ld, int H, float scale, hipStream_t stream, const char* name) {
  const int tiles = (int)((P + 31) / 32), smem = (H + 31) / 32 * (8 * kFrag * (int)sizeof(f16) + 2 * 32 * 4);
  const int grid = std::min((tiles + 3) / 4, 1024);   // four workgroups per CU
  KernelTimerScope timed(name, stream);
  hipLaunchKernelGGL(pair_bias_split_kernel, dim3((unsigned)grid), dim3(256), (unsigned)smem, stream, z, W, winv, wbias,
                     out, (unsigned)P, (unsigned)nrows, (unsigned)ncols, ld, H, scale, tiles);
  return check_launch(name);
}

}  // namespace bioemu
