// Pair-bias attention in fp32 on split f16 operands (split.h), head dim 24 or 32:
//   softmax(q k^T / sqrt(d) + bias; masked keys -> -1e6) v, gated by g.
//
//   kv_fragments_kernel  k and v of one (sequence, head, 32-key block) per wave -> operand
//                        fragments (8 KB) under one scale each, and the block's mask word.
//   attn_split_kernel    flash attention: a workgroup is 4 waves x 32 queries of one head; the
//                        waves share each block's fragments through LDS (copies that write it
//                        directly, double-buffered).
//
// Per block and wave: S^T = K Q^T (2 k-steps x 3 MFMAs; the head dim zero-padded to 32), online
// softmax in log2 units in registers, O^T = V^T P^T (2 x 3 MFMAs).  Lane (n, h) holds query n's
// logits of the keys 8 j + 4 h + t (register 4 j + t), which is the P operand of k-step ks when lane
// half h supplies the keys 16 ks + 4 h + 0..3 and 16 ks + 8 + 4 h + 0..3; V is stored with the same
// permutation.  The weights are below 2^14 times the running maximum's, which is their scale; a
// block's K and V scales are those of its unmasked keys alone (masked keys' logits are replaced and
// their weight is zero, so their rows are zeroed), and a block's O is added under its V scale.
// Blocks without an unmasked key are left out unless the sequence has none at all (then every
// weight is the same, as in softmax over equal logits).  Masked keys have a weight all the same where
// a query's every logit is near -1e6 or below: attend_all_keys computes such queries over all keys.
//
// 16 heads of 24, 768 tokens, 8 copies sharing one bias: 0.054 ms and 0.011 ms for the fragments, against 0.129 ms
// for the same flash form on fp32 MFMAs with per-key mask tests (28 MFMAs of 64 cycles and about 290 VALU
// instructions per block and wave; now 12 of 32 and about 130).  Bound by the VALU work of the softmax and the split
// of the weights.
#include "split.h"
#include "split_rows.h"

namespace bioemu {
namespace {

constexpr int kKvFrag = 4 * kFrag;             // f16: K k-steps 0, 1 | V k-steps 0, 1
constexpr float kMaskedLogit = -1e6f * kLog2e;
constexpr int kMaxBlocks = 4096;               // 32-key blocks of a sequence (the active list in LDS)

__device__ __forceinline__ float wave_absmax(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

// Wave per item (sequence bm, head, block kb).  kinv / vinv: 1 / scale per item; words: mask bits of block kb for
// each mask row (batch, or copy when mask_per_copy).
template <int HD>
__global__ __launch_bounds__(256) void kv_fragments_kernel(const float* __restrict__ k, const float* __restrict__ v,
                                                           const uint8_t* __restrict__ mask, f16* __restrict__ kv,
                                                           float* __restrict__ kvinv, uint32_t* __restrict__ words,
                                                           int N, int nkb, int H, int c_s, int mult, int mask_per_copy,
                                                           unsigned items) {
  const unsigned item = blockIdx.x * 4 + wave_id();
  if (item >= items) return;   // no barriers in this kernel
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const TileIdx t = split_tile(item, (unsigned)nkb, (unsigned)H);   // (bm, head, kb)
  const int bm = t.b, hd = t.row, kb = t.col, mrow = mask_per_copy ? bm : bm / mult;
  const int key = kb * 32 + n;
  const bool live = key < N;
  const unsigned word = (unsigned)__ballot(lane < 32 && live && mask[(size_t)mrow * N + min(key, N - 1)] != 0);
  if (hd == 0 && lane == 0 && (mask_per_copy || bm % mult == 0)) words[(size_t)mrow * nkb + kb] = word;
  const unsigned used = word ? word : (unsigned)__ballot(lane < 32 && live);
  const size_t row0 = (size_t)bm * N;
  float kk[2][8], vv[2][8];
  float ka = 0.f, va = 0.f;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int c = 16 * ks + 8 * h;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (c < HD && ((used >> n) & 1u)) {
      const float* p = k + (row0 + key) * c_s + hd * HD + c;
      a = *reinterpret_cast<const f32x4*>(p);
      b = *reinterpret_cast<const f32x4*>(p + 4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      kk[ks][e] = a[e];
      kk[ks][4 + e] = b[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int kx = 16 * ks + (e < 4 ? 4 * h + e : 8 + 4 * h + (e - 4));
      vv[ks][e] = 0.f;
      if (n < HD && ((used >> kx) & 1u)) vv[ks][e] = v[(row0 + kb * 32 + kx) * c_s + hd * HD + n];
      ka = fmaxf(ka, fabsf(kk[ks][e]));
      va = fmaxf(va, fabsf(vv[ks][e]));
    }
  }
  const float sk = split_scale(wave_absmax(ka)), sv = split_scale(wave_absmax(va));
  f16* d = kv + (size_t)item * kKvFrag + lane * 8;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    f16x8 kh, kl, vh, vl;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f16 x, y;
      split_value(kk[ks][e], sk, x, y);
      kh[e] = x;
      kl[e] = y;
      split_value(vv[ks][e], sv, x, y);
      vh[e] = x;
      vl[e] = y;
    }
    *reinterpret_cast<f16x8*>(d + ks * kFrag) = kh;
    *reinterpret_cast<f16x8*>(d + ks * kFrag + kFragHalf) = kl;
    *reinterpret_cast<f16x8*>(d + (2 + ks) * kFrag) = vh;
    *reinterpret_cast<f16x8*>(d + (2 + ks) * kFrag + kFragHalf) = vl;
  }
  if (lane == 0) {
    kvinv[2 * (size_t)item] = split_inv(sk);
    kvinv[2 * (size_t)item + 1] = split_inv(sv);
  }
}

// Query qr (one per lane pair) over all N keys in fp32, key by key; masked keys take part with logit -1e6.  Lane half h
// ends with the average's channels 8 j + 4 h + t in o[4 j + t] and the sum of the weights in l.  Slow, and reached only
// by queries that a masked key's weight matters to.
template <int HD>
__device__ __forceinline__ void attend_all_keys(const float* qr, const float* kb, const float* vb, const uint8_t* mask,
                                                const float* brow, int N, int c_s, float qscale, int h, float (&o)[16],
                                                float& l) {
  float q[HD];
#pragma unroll
  for (int c = 0; c < HD; ++c) q[c] = qr[c];
#pragma unroll
  for (int u = 0; u < 16; ++u) o[u] = 0.f;
  float m = -INFINITY, sum = 0.f;
  for (int j = 0; j < N; ++j) {
    float x = kMaskedLogit;
    if (mask[j]) {
      const float* kr = kb + (size_t)j * c_s;
      float dot = 0.f;
#pragma unroll
      for (int c = 0; c < HD; ++c) dot += q[c] * kr[c];
      x = dot * qscale + brow[j];
    }
    if (x == -INFINITY) continue;
    const float mn = fmaxf(m, x), alpha = fast_exp2(m - mn), p = fast_exp2(x - mn);   // alpha 0 at the first key
    const float* vr = vb + (size_t)j * c_s;
    sum = sum * alpha + p;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int c = 8 * (u >> 2) + 4 * h + (u & 3);
      if (8 * (u >> 2) < HD) o[u] = o[u] * alpha + p * vr[c];
    }
    m = mn;
  }
  l = sum;
}

// bias [B][H][N][ld] in log2 units; k, v and mask as kv_fragments_kernel's.
template <int HD>
__global__ __launch_bounds__(256, 3) void attn_split_kernel(const float* __restrict__ q, const f16* __restrict__ kv,
                                                            const float* __restrict__ kvinv,
                                                            const uint32_t* __restrict__ words,
                                                            const float* __restrict__ g, const float* __restrict__ bias,
                                                            const float* __restrict__ k, const float* __restrict__ v,
                                                            const uint8_t* __restrict__ mask,
                                                            float* __restrict__ go, int N, int nkb, int ld, int H,
                                                            int c_s, int mult, float qscale, int mask_per_copy,
                                                            int nqb, int total) {
  __shared__ __attribute__((aligned(16))) f16 smem[2][kKvFrag];
  __shared__ uint16_t active[kMaxBlocks];
  __shared__ int nactive, nvalid;   // nvalid: whether a key is valid
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 31, h = lane >> 5;
  // an XCD takes consecutive items, the copies that share a bias block next to each other
  const int per_xcd = (total + 7) / 8, item = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (item >= total || (int)(blockIdx.x / 8) >= per_xcd) return;   // uniform over the workgroup
  const int copy = item % mult, r = item / mult, qb = r % nqb, bh = r / nqb, hd = bh % H, b = bh / H;
  const int bm = b * mult + copy;
  const uint32_t* wrow = words + (size_t)(mask_per_copy ? bm : b) * nkb;
  if (wave == 0) {
    bool some = false;
    for (int k0 = 0; k0 < nkb; k0 += 64) some |= __any(k0 + lane < nkb && wrow[min(k0 + lane, nkb - 1)] != 0);
    int count = 0;
    for (int k0 = 0; k0 < nkb; k0 += 64) {
      const bool on = k0 + lane < nkb && (!some || wrow[min(k0 + lane, nkb - 1)] != 0);
      const unsigned long long m = __ballot(on);
      if (on) active[count + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)(k0 + lane);
      count += __popcll(m);
    }
    if (lane == 0) {
      nactive = count;
      nvalid = some;
    }
  }
  const int q0 = (qb * 4 + wave) * 32;
  // waves past N run on a clamped row and store nothing: they copy their share of every block and meet every barrier
  const int qi = min(q0 + n, N - 1);
  SplitFrag qf[2];
  float qinv;
  {
    const float* qr = q + ((size_t)bm * N + qi) * c_s + hd * HD;
    float v[2][8];
    float amax = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int c = 16 * ks + 8 * h;
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
      if (c < HD) {
        x = *reinterpret_cast<const f32x4*>(qr + c);
        y = *reinterpret_cast<const f32x4*>(qr + c + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[ks][e] = x[e];
        v[ks][4 + e] = y[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[ks][e]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    const float s = split_scale(amax);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        f16 x, y;
        split_value(v[ks][e], s, x, y);
        qf[ks].hi[e] = x;
        qf[ks].lo[e] = y;
      }
    qinv = split_inv(s) * qscale;   // logits in log2 units
  }
  const size_t item0 = ((size_t)bm * H + hd) * nkb;
  const float* brow = bias + (((size_t)b * H + hd) * N + qi) * ld + 4 * h;
  auto stage = [&](int kb, int st) {
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(kv + (item0 + kb) * kKvFrag, kKvFrag * 2);
#pragma unroll
    for (int p = 0; p < 2; ++p)
      copy1k_to_lds(rs, &smem[st][(wave * 2 + p) * kFragHalf], lane * 16, (unsigned)(wave * 2 + p) * 1024);
  };
  auto load_bias = [&](int kb, f32x4 (&bb)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) bb[j] = *reinterpret_cast<const f32x4*>(brow + kb * 32 + 8 * j);
  };
  __syncthreads();   // the active list
  const int na = nactive;
  int kb = __builtin_amdgcn_readfirstlane(active[0]);
  f32x4 bb[4];
  stage(kb, 0);
  load_bias(kb, bb);
  f32x16 o = zero16();
  float m = -INFINITY, l = 0.f;
#pragma unroll 1
  for (int a = 0; a < na; ++a) {
    const int st = a & 1;
    const unsigned word = wrow[kb];
    const float sk = kvinv[2 * (item0 + kb)] * qinv, sv = kvinv[2 * (item0 + kb) + 1];
    const int kcur = kb;
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies (and bias loads) of the block landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
    const f16* f = smem[st];
    SplitFrag kf[2], vf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) kf[ks] = load_frag(f + ks * kFrag, lane);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) vf[ks] = load_frag(f + (2 + ks) * kFrag, lane);
    const int nk = a + 1 < na ? __builtin_amdgcn_readfirstlane(active[a + 1]) : kb;
    // every LDS read of the block precedes the next block's copies: the compiler makes a later one wait for them
    __builtin_amdgcn_sched_barrier(0);
    f32x4 bn[4];
    if (a + 1 < na) {
      kb = nk;
      stage(kb, st ^ 1);
      load_bias(kb, bn);
    }
    f32x16 s = zero16();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) mfma_split(kf[ks], qf[ks], s);
    float x[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = s[u] * sk + bb[u >> 2][u & 3];
    if (word != 0xffffffffu) {   // a masked key, or keys past N
      const unsigned w = word >> (4 * h);
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int kx = 8 * (u >> 2) + (u & 3);
        x[u] = (w >> kx) & 1u ? x[u] : (kcur * 32 + kx + 4 * h < N ? kMaskedLogit : -INFINITY);
      }
    }
    float bmax = x[0];
#pragma unroll
    for (int u = 1; u < 16; ++u) bmax = fmaxf(bmax, x[u]);
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32));
    if (__any(bmax > m)) {
      const float mn = fmaxf(m, bmax), alpha = fast_exp2(m - mn);   // 0 at the first block (m = -inf)
      l *= alpha;
#pragma unroll
      for (int u = 0; u < 16; ++u) o[u] *= alpha;
      m = mn;
    }
    const float mm = m - 14.f;   // weights times 2^14
    SplitFrag pf[2];
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float p = fast_exp2(x[u] - mm);
      sum += p;
      f16 c, d;
      split_value(p, 1.0f, c, d);
      pf[u >> 3].hi[u & 7] = c;
      pf[u >> 3].lo[u & 7] = d;
    }
    l += sum;
    f32x16 ob = zero16();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) mfma_split(vf[ks], pf[ks], ob);
#pragma unroll
    for (int u = 0; u < 16; ++u) o[u] += ob[u] * sv;
#pragma unroll
    for (int j = 0; j < 4; ++j) bb[j] = bn[j];
  }
  l += __shfl_xor(l, 32);
  if (q0 + n >= N) return;
  if (nvalid && m < kMaskedLogit + 160.f) {   // a masked key's weight is not zero
    const size_t row0 = (size_t)bm * N * c_s + hd * HD;
    float oa[16];
    attend_all_keys<HD>(q + row0 + (size_t)qi * c_s, k + row0, v + row0, mask + (size_t)(mask_per_copy ? bm : b) * N,
                        brow - 4 * h, N, c_s, qscale, h, oa, l);
#pragma unroll
    for (int u = 0; u < 16; ++u) o[u] = oa[u];
  }
  const float inv = 1.0f / l;
  const size_t off = ((size_t)bm * N + qi) * c_s + hd * HD;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = 8 * j + 4 * h;
    if (c < HD) {
      const f32x4 gv = *reinterpret_cast<const f32x4*>(g + off + c);
      f32x4 rr;
#pragma unroll
      for (int t = 0; t < 4; ++t) rr[t] = gv[t] * (o[4 * j + t] * inv);
      *reinterpret_cast<f32x4*>(go + off + c) = rr;
    }
  }
}

template <int HD>
int launch(const SplitAttn& a, hipStream_t stream, const char* name) {
  const int nkb = (a.N + 31) / 32, nqb = (a.N + 127) / 128;
  const long long items = (long long)a.BM * a.H * nkb, total = (long long)a.BM * a.H * nqb;
  if (nkb > kMaxBlocks || items >= (1LL << 31) || total >= (1LL << 28))
    return set_error(BIOEMU_ERR_UNSUPPORTED, "%s: too many keys or sequences (N=%d, %d sequences)", name, a.N, a.BM);
  {
    KernelTimerScope timed("f32_kv_fragments", stream);
    hipLaunchKernelGGL(kv_fragments_kernel<HD>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, stream, a.k, a.v,
                       a.mask, a.kv, a.kvinv, a.words, a.N, nkb, a.H, a.c_s, a.mult, a.mask_per_copy, (unsigned)items);
  }
  const int rc = check_launch("f32_kv_fragments");
  if (rc) return rc;
  KernelTimerScope timed(name, stream);
  const float qscale = kLog2e / sqrtf((float)HD);
  hipLaunchKernelGGL(attn_split_kernel<HD>, dim3((unsigned)((total + 7) / 8 * 8)), dim3(256), 0, stream, a.q, a.kv,
                     a.kvinv, a.words, a.g, a.bias, a.k, a.v, a.mask, a.go, a.N, nkb, a.ld, a.H, a.c_s, a.mult, qscale,
                     a.mask_per_copy,
                     nqb, (int)total);
  return check_launch(name);
}

}  // namespace

size_t split_attn_kv_elems(int64_t BM, int64_t H, int64_t N) { return (size_t)(BM * H * ((N + 31) / 32)) * kKvFrag; }

int split_attn(const SplitAttn& a, hipStream_t stream, const char* name) {
  return a.c_s / a.H == 24 ? launch<24>(a, stream, name) : launch<32>(a, stream, name);
}

}  // namespace bioemu
