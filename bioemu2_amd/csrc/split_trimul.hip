// Triangle multiplicative update in fp32 on split f16 operands (split.h), 128 channels
// (TriangleMultiplicationFull.forward, src/bioemu2/biomoa/ops/triangle_multiplication.py:89-99):
//
//   trimul_planes_kernel    LN(x) -> (p, g) -> p * sigmoid(g) * mask, written channel-major as
//                           hi and lo planes [channel][i][k] (k = r2 outgoing, r1 incoming), so
//                           that both directions contract C = A B^T with k contiguous.  A plane's
//                           scale is a bound from its weights (|p sigmoid(g)| <= |p|,
//                           SplitMat::norm), so it is known before the first row is seen.
//                           32 pairs of a line that are all below 2^-12 of that range take
//                           a power of two more (their gain, one byte); a channel with
//                           such a line is flagged.
//   trimul_contract_kernel  o[d][i][j] = sum_k a[d][i][k] b[d][j][k] on 128 x 128 tiles;
//                           gains of a flagged channel are undone 32 k at a time (a wave
//                           sums 32 k that hold one by themselves: there the last bits of
//                           its 64 x 64 block depend on its other rows' gains).
//   trimul_out_kernel       LN_out(o) Wp * sigmoid(LN_in(x) Wg) (+ x): o read from its planes,
//                           32 pairs (128 bytes) of a channel per load, both weights resident in LDS.
//
// LayerNorm affines are folded into the weights that follow (SplitMat::gamma).
//
// N = 333, against the fp32-MFMA kernels these replace (operands from L2, the contraction stored 4 bytes at a time
// pair-major, LayerNorms and the gate through memory): projection 0.079 ms (was 0.283, with 0.030 of zero fill and
// 0.042 of LayerNorm), contraction 0.054 (0.376; 174 TFLOP/s of fp32 products on the padded 384 x 384 x 352, bound by
// LDS like split_gemm_kernel), output 0.055 (0.226, with 0.042 of LayerNorm and 0.067 of gate).  The sigmoids
// keep an ulp's accuracy: with the plain hardware exp2 and reciprocal the result was 1.4 times as far from float64.
#include <algorithm>
#include <type_traits>

#include "split.h"
#include "split_rows.h"

namespace bioemu {
namespace {

constexpr int D = 128;
constexpr int kWBlock = 8 * kFrag;   // f16 elements: a 32 x 128 weight block

// Row stride (f16 or fp32 elements) of a plane: N columns, zero-filled to whole 32-wide k-steps.
__host__ __device__ inline int plane_ld(int N) { return (N + 31) / 32 * 32; }

// Gains: bytes [channel plane][32-k tile][row, plane_ld], 2^gain the factor; row tiles read past the last row.
__host__ __device__ inline size_t gain_at(size_t plane, int kt, int i, int ld) {
  return (plane * (ld / 32) + kt) * ld + i;
}
constexpr int kGainPad = 128;
constexpr float kGainBelow = 8.f;   // scaled magnitude

__global__ __launch_bounds__(256, 2) void trimul_planes_kernel(const float* __restrict__ x,
                                                               const uint8_t* __restrict__ mask,
                                                               const f16* __restrict__ W,
                                                               const float* __restrict__ winv,
                                                               const float* __restrict__ wnorm,
                                                               const float* __restrict__ wbias, f16* __restrict__ hi,
                                                               f16* __restrict__ lo, uint8_t* __restrict__ gains,
                                                               uint32_t* __restrict__ flags, int N, int outgoing,
                                                               unsigned tiles, int per) {
  __shared__ __attribute__((aligned(16))) f16 smem[2][2 * kWBlock];   // p | g block, double-buffered: 64 KB
  __shared__ float sbias[4 * D], swinv[4 * D];   // swinv: [column block][p | g][32], as the weights
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(W, 8 * 2 * kWBlock * 2);
  auto stage = [&](int cb) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int c = wave * 8 + q;
      copy1k_to_lds(rw, &smem[cb & 1][c * kFragHalf], lane * 16, (unsigned)(cb * 2 * kWBlock * 2 + c * 1024));
    }
  };
  const int first = blockIdx.y * per, last = first + per;   // this workgroup's column blocks
  stage(first);
  stage_floats(sbias, wbias, 4 * D, 4 * D);
  stage_floats(swinv, winv, 4 * D, 4 * D, 1.0f / kNormScale);
  // tile (b, i, kb): 32 pairs k = 32 kb .. of line i; a wave past the last tile works on tile 0 and stores nothing
  const unsigned tile = blockIdx.x * 4 + wave;
  const bool live = tile < tiles;
  const int ld = plane_ld(N), kbs = ld / 32;
  const TileIdx t = split_tile(live ? tile : 0, (unsigned)kbs, (unsigned)N);
  const int i = t.row, k0 = t.col * 32;
  const size_t b0 = (size_t)t.b * N * N;
  auto pair = [&](int k) { return b0 + (outgoing ? (size_t)i * N + k : (size_t)k * N + i); };
  const unsigned long long kept = __ballot(lane < 32 && k0 + lane < N && mask[pair(min(k0 + lane, N - 1))] != 0);
  SplitFrag xf[8];
  float xinv;   // of pair perm32(n)
  {
    float v[64];
    load_row_half<D>(x + pair(min(k0 + perm32(n), N - 1)) * D, h, v);
    xinv = normalized_row_half<D>(v, xf);
  }
  const bool scaled_rows = __any(xinv != 1.0f);
  const unsigned keep = (unsigned)kept >> (16 * h);   // bit u: pair 16 h + u
  const size_t plane = (size_t)N * ld;
#pragma unroll 1
  for (int cb = first; cb < last; ++cb) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of block cb landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
    if (cb + 1 < last) stage(cb + 1);
    // pair slots are the MFMA rows (in perm32 order), channels its columns: lane (n, h) ends with the 16
    // consecutive pairs 16 h + u of channel perm32(n)
    const f16* st = smem[cb & 1];
    f32x16 p = zero16(), g = zero16();
    mfma_block2<8, false>(st, st + kWBlock, xf, xf, lane, p, g);
    if (scaled_rows) {   // register u is pair 16 h + u, whose row lane 8 (u / 4) + 4 h + u % 4 holds
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float xi = __shfl(xinv, 8 * (u >> 2) + 4 * h + (u & 3));
        p[u] *= xi;
        g[u] *= xi;
      }
    }
    const int c = cb * 32 + perm32(n);
    const int cw = cb * 64 + perm32(n);
    const float sp = swinv[cw], sg = swinv[cw + 32];
    const float bp = sbias[c], bg = sbias[2 * D + c];
    float s = split_scale(wnorm[cw] * 1.01f), v[16], amax = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      v[u] = (keep >> u) & 1u ? (p[u] * sp + bp) * sigmoid_ulp(g[u] * sg + bg) : 0.f;
      amax = fmaxf(amax, fabsf(v[u]));
    }
    amax = max_halves(amax);
    const bool low = amax * s < kGainBelow && amax > 0.f;
    if (__any(low)) {
      const float s2 = low ? split_scale(amax) : s;
      if (low && live && h == 0) {
        const size_t ch = (size_t)t.b * 2 * D + c;
        gains[gain_at(ch, t.col, i, ld)] =
            (uint8_t)((__builtin_bit_cast(uint32_t, s2) >> 23) - (__builtin_bit_cast(uint32_t, s) >> 23));
        flags[ch] = 1;
      }
      s = s2;
    }
    f16x8 vh[2], vl[2];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      f16 a, d;
      split_value(v[u], s, a, d);
      vh[u >> 3][u & 7] = a;
      vl[u >> 3][u & 7] = d;
    }
    if (live) {
      const size_t off = ((size_t)t.b * 2 * D + c) * plane + (size_t)i * ld + k0 + 16 * h;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        *reinterpret_cast<f16x8*>(hi + off + 8 * q) = vh[q];
        *reinterpret_cast<f16x8*>(lo + off + 8 * q) = vl[q];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Contraction: 4 waves of 64 x 64, 32 k per stage: hi and lo of 128 rows of A and of B, 64-byte rows whose four
// 16-byte chunks are XOR-swizzled (rows r, r + 4, r + 8, r + 12 share a bank group base), double-buffered.
// ---------------------------------------------------------------------------
constexpr int kPart = 128 * 32;      // f16 elements of one staged plane tile: 8 KB
constexpr int kCStage = 4 * kPart;   // A hi | A lo | B hi | B lo
constexpr int kCSmem = 2 * kCStage * (int)sizeof(f16);   // 64 KB: two workgroups per CU

__device__ __forceinline__ int swz(int r) { return (r >> 2) & 3; }

__global__ __launch_bounds__(256, 2) void trimul_contract_kernel(const f16* __restrict__ hi,
                                                                 const f16* __restrict__ lo,
                                                                 const float* __restrict__ wnorm,
                                                                 const uint8_t* __restrict__ gains,
                                                                 const uint32_t* __restrict__ flags,
                                                                 float* __restrict__ o, int N, int nt, int total) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f16* smem = reinterpret_cast<f16*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  const int wi = wave & 1, wj = wave >> 1;
  // an XCD takes consecutive tiles: a plane's tiles share its L2
  const int per_xcd = (total + 7) / 8, item = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (item >= total || (int)(blockIdx.x / 8) >= per_xcd) return;   // uniform over the workgroup
  const int z = item / (nt * nt), r = item % (nt * nt), it = r / nt, jt = r % nt;
  const int b = z / D, d = z % D;
  const int ld = plane_ld(N);
  const size_t plane = (size_t)N * ld;
  const size_t pa = ((size_t)b * 2 * D + d) * plane + (size_t)it * 128 * ld;
  const size_t pb = ((size_t)b * 2 * D + D + d) * plane + (size_t)jt * 128 * ld;
  // rows past N read as zeros through the buffer bounds
  const unsigned ba = (unsigned)min(N - it * 128, 128) * ld * 2, bb = (unsigned)min(N - jt * 128, 128) * ld * 2;
  const __amdgpu_buffer_rsrc_t rs[4] = {buffer_rsrc(hi + pa, ba), buffer_rsrc(lo + pa, ba), buffer_rsrc(hi + pb, bb),
                                        buffer_rsrc(lo + pb, bb)};
  unsigned vo[2];   // wave w copies rows 32 w .. + 31 of each part, 16 rows (1 KB) at a time
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = wave * 32 + q * 16 + (lane >> 2);
    vo[q] = (unsigned)(row * ld + ((lane & 3) ^ swz(row)) * 8) * 2;
  }
  auto stage = [&](int kt) {
    f16* st = smem + (kt & 1) * kCStage;
#pragma unroll
    for (int part = 0; part < 4; ++part)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        copy1k_to_lds(rs[part], st + part * kPart + (wave * 2 + q) * 512, vo[q], (unsigned)kt * 64);
  };
  f32x16 acc[2][2];   // [i block][j block]
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = zero16();
  const int nk = ld / 32;
  const size_t cha = (size_t)b * 2 * D + d, chb = cha + D;
  const bool flagged = flags[cha] | flags[chb];   // uniform over the workgroup
  stage(0);
  auto run = [&](auto gained) {   // two loops: the one without gains is free of their registers and branches
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of the stage landed
      __syncthreads();                       // ... and everyone's; the other stage is free again
      if (kt + 1 < nk) stage(kt + 1);
      const f16* st = smem + (kt & 1) * kCStage;
      SplitFrag fa[2][2], fb[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int ra = wi * 64 + x * 32 + n, rb = wj * 64 + x * 32 + n;
          const int oa = (ra * 4 + ((2 * ks + h) ^ swz(ra))) * 8, ob = (rb * 4 + ((2 * ks + h) ^ swz(rb))) * 8;
          fa[ks][x].hi = *reinterpret_cast<const f16x8*>(st + oa);
          fa[ks][x].lo = *reinterpret_cast<const f16x8*>(st + kPart + oa);
          fb[ks][x].hi = *reinterpret_cast<const f16x8*>(st + 2 * kPart + ob);
          fb[ks][x].lo = *reinterpret_cast<const f16x8*>(st + 3 * kPart + ob);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (gained.value) {
        uint32_t ga[2][4], some = 0;   // ga: four rows each
        int gb[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int row = it * 128 + wi * 64 + x * 32 + 8 * q + 4 * h;
            ga[x][q] = *reinterpret_cast<const uint32_t*>(gains + gain_at(cha, kt, row, ld));
            some |= ga[x][q];
          }
          gb[x] = gains[gain_at(chb, kt, jt * 128 + wj * 64 + x * 32 + n, ld)];
          some |= gb[x];
        }
        if (__any(some != 0)) {
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
              f32x16 part = zero16();
#pragma unroll
              for (int ks = 0; ks < 2; ++ks) mfma_split(fa[ks][x], fb[ks][y], part);
#pragma unroll
              for (int u = 0; u < 16; ++u)
                acc[x][y][u] +=
                    __builtin_amdgcn_ldexpf(part[u], -((int)(ga[x][u >> 2] >> (8 * (u & 3)) & 0xffu) + gb[y]));
            }
          continue;
        }
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) mfma_split(fa[ks][x], fb[ks][y], acc[x][y]);
    }
  };
  if (flagged)
    run(std::true_type{});
  else
    run(std::false_type{});
  // lane n: column j, register u: row 8 (u / 4) + 4 h + u % 4; a store covers 128 bytes of two rows
  const int dw = d / 32 * 64 + d % 32;   // channel d's place among the p rows' norms
  const float s = split_inv(split_scale(wnorm[dw] * 1.01f)) * split_inv(split_scale(wnorm[dw + 2 * D] * 1.01f));
  float* po = o + ((size_t)b * D + d) * plane;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int i0 = it * 128 + wi * 64 + x * 32 + 4 * h, j = jt * 128 + wj * 64 + y * 32 + n;
      if (j >= ld) continue;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int i = i0 + 8 * (u >> 2) + (u & 3);
        if (i < N) po[(size_t)i * ld + j] = acc[x][y][u] * s;
      }
    }
}

// ---------------------------------------------------------------------------
// Output: a wave per 32 pairs (i, j0 .. j0 + 31) of a line, or (kFew) a workgroup of four waves, each of which
// normalises the pairs and takes one of the four column blocks.
// ---------------------------------------------------------------------------
constexpr int kOutWaves = 8;

// p * sigmoid(g), rounded by itself: the residual add that follows is the same sum a caller would make.
__device__ __forceinline__ float gated(float p, float g) {
#pragma clang fp contract(off)
  return p * sigmoid_ulp(g);
}
constexpr int kOutWeights = 2 * 4 * kWBlock;                                  // f16: p_out | g_out
constexpr int kOutSmem = kOutWeights * (int)sizeof(f16) + 4 * D * 4;   // 128 KB, the biases and the weights' scales

template <bool kFew>
__global__ __launch_bounds__(64 * (kFew ? 4 : kOutWaves), kFew ? 1 : 2) void trimul_out_kernel(
    const float* x, const float* __restrict__ o, const f16* __restrict__ W, const float* __restrict__ winv,
    const float* __restrict__ wbias, float* out, int N, int residual, unsigned tiles) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  f16* smem = reinterpret_cast<f16*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  float* sbias = reinterpret_cast<float*>(smem + kOutWeights);
  float* swinv = sbias + 2 * D;
  stage_floats(sbias, wbias, 2 * D, 2 * D);
  stage_floats(swinv, winv, 2 * D, 2 * D, 1.0f / kNormScale);
  if (kFew) {   // this wave's two weight blocks; waited for below the rows' loads
    const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(W, kOutWeights * 2);
#pragma unroll
    for (int c = 0; c < 32; ++c) {
      const int at = (c < 16 ? wave : 4 + wave) * 16 + c % 16;
      copy1k_to_lds(rw, smem + at * kFragHalf, lane * 16, (unsigned)at * 1024);
    }
  } else {
    stage_fragments(W, smem, kOutWeights / kFragHalf, kOutWaves, wave, lane);
  }
  const int ld = plane_ld(N);
  const size_t plane = (size_t)N * ld;
#pragma unroll 1
  for (unsigned tile = kFew ? blockIdx.x : blockIdx.x * kOutWaves + wave; tile < tiles;
       tile += gridDim.x * (kFew ? 1 : kOutWaves)) {
    const TileIdx t = split_tile(tile, (unsigned)(ld / 32), (unsigned)N);
    const int j = t.col * 32 + n;
    const bool valid = j < N;
    const size_t m = ((size_t)t.b * N + t.row) * N + min(j, N - 1);
    SplitFrag of[8], xf[8];
    float oinv, xinv;
    {
      float v[64];
      const float* po = o + ((size_t)t.b * D + 8 * h) * plane + (size_t)t.row * ld + j;
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[8 * s + e] = po[(size_t)(16 * s + e) * plane];
      oinv = normalized_row_half<D>(v, of);
    }
    {
      float v[64];
      load_row_half<D>(x + m * D, h, v);
      xinv = normalized_row_half<D>(v, xf);
    }
    if (kFew) {   // every wave holds the rows before one overwrites them
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
    }
#pragma unroll 1
    for (int cb = kFew ? wave : 0; cb < (kFew ? wave + 1 : 4); ++cb) {
      const f16* w = smem + cb * kWBlock;
      f32x16 p = zero16(), g = zero16();
      mfma_block2<8>(w, w + 4 * kWBlock, of, xf, lane, p, g);
      undo_gain(p, oinv);
      undo_gain(g, xinv);
      const int c = cb * 32 + 16 * h;
      if (valid) {
        f32x4 xr[4];   // read ahead of the stores (out may be x)
        if (residual)
#pragma unroll
          for (int q = 0; q < 4; ++q) xr[q] = *reinterpret_cast<const f32x4*>(x + m * D + c + 4 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 bp = *reinterpret_cast<const f32x4*>(sbias + c + 4 * q);
          const f32x4 bg = *reinterpret_cast<const f32x4*>(sbias + D + c + 4 * q);
          const f32x4 wp = *reinterpret_cast<const f32x4*>(swinv + c + 4 * q);
          const f32x4 wg = *reinterpret_cast<const f32x4*>(swinv + D + c + 4 * q);
          f32x4 r;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r[e] = gated(p[4 * q + e] * wp[e] + bp[e], g[4 * q + e] * wg[e] + bg[e]);
          if (residual) {
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] += xr[q][e];
          }
          *reinterpret_cast<f32x4*>(out + m * D + c + 4 * q) = r;
        }
      }
    }
  }
}

// Workspace: weight fragments and their scales, the hi and lo planes, o.
struct Layout {
  size_t win, wout, scales, gains, flags, gain_bytes, hi, lo, o, total;
};
Layout layout(int64_t B, int64_t N) {
  Layout L;
  const size_t plane = (size_t)N * plane_ld((int)N);
  size_t off = 0;
  auto take = [&](size_t n) {
    const size_t at = off;
    off += (size_t)round_up((int64_t)n, 256);
    return at;
  };
  L.win = take((size_t)16 * kWBlock * 2);
  L.wout = take((size_t)8 * kWBlock * 2);
  L.scales = take((4 * D + 4 * D + 2 * D + 4 * D + 2 * D) * 4);
  L.gains = off;   // and the flags, cleared together
  L.flags = L.gains + (size_t)round_up((int64_t)gain_at((size_t)B * 2 * D, 0, 0, plane_ld((int)N)) + kGainPad, 16);
  L.gain_bytes = L.flags + (size_t)B * 2 * D * 4 - L.gains;
  take(L.gain_bytes);
  L.hi = take((size_t)B * 2 * D * plane * 2);
  L.lo = take((size_t)B * 2 * D * plane * 2);
  L.o = take((size_t)B * D * plane * 4);
  L.total = off;
  return L;
}

}  // namespace

size_t split_trimul_workspace_bytes(int64_t B, int64_t N) { return layout(B, N).total; }

int split_trimul(const float* x, const uint8_t* mask, const float* norm_in_w, const float* norm_in_b,
                 const float* p_in_w, const float* g_in_w, const float* norm_out_w, const float* norm_out_b,
                 const float* p_out_w, const float* g_out_w, float* out, void* workspace, int64_t B, int64_t N,
                 int outgoing, int residual, hipStream_t stream) {
  const Layout L = layout(B, N);
  char* base = static_cast<char*>(workspace);
  f16 *win = reinterpret_cast<f16*>(base + L.win), *wout = reinterpret_cast<f16*>(base + L.wout);
  f16 *hi = reinterpret_cast<f16*>(base + L.hi), *lo = reinterpret_cast<f16*>(base + L.lo);
  float* o = reinterpret_cast<float*>(base + L.o);
  float *inv_in = reinterpret_cast<float*>(base + L.scales), *norm_in = inv_in + 4 * D,
        *inv_out = norm_in + 4 * D, *bias_in = inv_out + 2 * D, *bias_out = bias_in + 4 * D;
  SplitMats mats{};
  mats.m[0] = with_fold(split_gemm_weight(p_in_w, win, inv_in, norm_in, 2 * D, D, 2, 0), norm_in_w, norm_in_b, bias_in);
  mats.m[1] =
      with_fold(split_gemm_weight(g_in_w, win, inv_in, norm_in, 2 * D, D, 2, 1), norm_in_w, norm_in_b, bias_in + 2 * D);
  mats.m[2] = with_fold(split_gemm_weight(p_out_w, wout, inv_out, nullptr, D, D), norm_out_w, norm_out_b, bias_out);
  mats.m[3] = with_fold(split_gemm_weight(g_out_w, wout + 4 * kWBlock, inv_out + D, nullptr, D, D), norm_in_w,
                        norm_in_b, bias_out + D);
  uint8_t* gains = reinterpret_cast<uint8_t*>(base + L.gains);
  uint32_t* flags = reinterpret_cast<uint32_t*>(base + L.flags);
  mats.zero = gains;
  mats.zero_bytes = L.gain_bytes;
  int rc = split_weights(mats, 4, stream);
  if (rc) return rc;
  const unsigned tiles = (unsigned)(B * N * (plane_ld((int)N) / 32));
  {
    // As many parts of the eight column blocks as make one round of two workgroups per CU.  The call, all blocks / these
    // parts (us): N = 40 48 / 31, N = 64 52 / 33, N = 100 69 / 56, N = 160 72 / 65; two rounds: 31, 34, 59, 70.
    const unsigned wgs = (tiles + 3) / 4, resident = 2u * compute_units();
    unsigned parts = 1;
    while (parts < 8 && 2 * parts * wgs <= resident) parts *= 2;
    KernelTimerScope timed("f32_trimul_proj", stream);
    hipLaunchKernelGGL(trimul_planes_kernel, dim3(wgs, parts), dim3(256), 0, stream, x, mask, win, inv_in, norm_in,
                       bias_in, hi, lo, gains, flags, (int)N, outgoing, tiles, 8 / (int)parts);
  }
  if ((rc = check_launch("f32_trimul_proj"))) return rc;
  {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(trimul_contract_kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kCSmem);
    if (e != hipSuccess) return set_error(BIOEMU_ERR_LAUNCH, "f32_trimul_contract: %s", hipGetErrorString(e));
    const int nt = (int)((N + 127) / 128), total = (int)(B * D) * nt * nt;
    KernelTimerScope timed("f32_trimul_contract", stream);
    hipLaunchKernelGGL(trimul_contract_kernel, dim3((unsigned)((total + 7) / 8 * 8)), dim3(256), kCSmem, stream, hi, lo,
                       norm_in, gains, flags, o, (int)N, nt, total);
  }
  if ((rc = check_launch("f32_trimul_contract"))) return rc;
  {
    const unsigned cus = compute_units();
    // One round of a tile a workgroup (the call, us, a tile a wave / a workgroup: N = 40 38 / 31, N = 64 41 / 33, N = 80,
    // 240 tiles, 48 / 40; N = 100, 400 tiles, 54 / 56, N = 160, 800 tiles, 65 / 88).
    const bool few = tiles <= cus;
    const auto kernel = few ? trimul_out_kernel<true> : trimul_out_kernel<false>;
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kOutSmem);
    if (e != hipSuccess) return set_error(BIOEMU_ERR_LAUNCH, "f32_trimul_out: %s", hipGetErrorString(e));
    const unsigned grid = few ? tiles : std::min((tiles + kOutWaves - 1) / kOutWaves, cus);
    KernelTimerScope timed("f32_trimul_out", stream);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * (few ? 4 : kOutWaves)), kOutSmem, stream, x, o, wout, inv_out,
                       bias_out, out, (int)N, residual, tiles);
  }
  return check_launch("f32_trimul_out");
}

}  // namespace bioemu
