// Batched bf16 NT GEMM on MFMA: C[z][i][j] = sum_k A[z][i][k] * B[z][j][k].
//
// Used for the per-channel triangle contraction, where both operands are
// channel-major [z = b*D + d][row][k] planes with k contiguous: n rows of
// stride ld = n rounded up to 64, zero-filled past n, so that the reduction
// runs over whole 64-wide k-tiles.  Rows past n read as zero through the
// buffer bounds; C has the same layout (its columns in [n, ld) come out zero).
//
// Two tilings of the same k order (so the same result bits): 256 x 256 with
// the k-tile body of gemm_nt.h (8 waves), and 128 x 128 (4 waves of 64 x 64,
// two workgroups per CU) for sizes that leave the large tiles mostly padding
// or most CUs without one; BK = 64, staged into LDS by direct copies.
//
// The 256 x 256 kernel is persistent: one workgroup per CU walks a list of
// tiles.  Tile rounds in lock-step end in synchronized bursts (every CU stores
// its 128 KB tile, then every CU waits for its next tile's first k-tile); here
// the next tile's first k-tile is requested during the current tile's last
// k-tile, so it is in flight while the current tile is stored.  The tiles are
// dealt per XCD (workgroup w runs on XCD w % 8): XCD x owns a contiguous range
// of tiles, its workgroups take them round-robin, so the tiles of one plane,
// which read the same rows, run together on one L2.  (Splitting the tiles left
// over after even rounds into 256 x 128 halves, dealt first to half the
// workgroups and last to the others, measured slower at N = 768: 0.177 vs
// 0.168 ms.)  A wave whose 64 x 128 block lies past n skips its products.
#include "common.h"
#include "gemm_nt.h"
#include "internal.h"
#include "pairtile.h"

namespace bioemu {
namespace {

__global__ __launch_bounds__(kNtThreads) void bgemm_nt_kernel(const bf16* __restrict__ A, const bf16* __restrict__ B,
                                                              bf16* __restrict__ C, int n, int ld, int total,
                                                              int nwg) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  bf16* smem = reinterpret_cast<bf16*>(smem_raw);
  const int tpr = (n + kNtTile - 1) / kNtTile, tiles = tpr * tpr;
  const size_t plane = (size_t)n * ld;
  // this workgroup's tiles: t = first + l, first + l + L, ... < last
  const int xcd = blockIdx.x % kNtXcds, l = blockIdx.x / kNtXcds, L = nwg / kNtXcds;
  const int per_xcd = (total + kNtXcds - 1) / kNtXcds;
  const int first = xcd * per_xcd, last = min(total, first + per_xcd);
  int t = first + l;
  if (t >= last) return;   // the whole workgroup, before any barrier

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, lh = lane >> 5;
  const int wi = wave & 3, wj = wave >> 2;
  const NtStaging stg(wave, lane, ld, kNtTile);
  int offj[4], offi[2];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) offj[jb] = wj * 128 + jb * 32 + perm32(ln);
#pragma unroll
  for (int ib = 0; ib < 2; ++ib) offi[ib] = wi * 64 + ib * 32 + ln;
  auto rsrc = [&](const bf16* M, int z, int rt) {
    return buffer_rsrc(M + z * plane + (size_t)rt * kNtTile * ld, (unsigned)min(n - rt * kNtTile, kNtTile) * ld * 2);
  };
  auto a_rsrc = [&](int tt) { return rsrc(A, tt / tiles, tt % tiles / tpr); };
  auto b_rsrc = [&](int tt) { return rsrc(B, tt / tiles, tt % tiles % tpr); };
  const int nk = ld / kNtBK;
  __amdgpu_buffer_rsrc_t ra = a_rsrc(t), rb = b_rsrc(t);
  stg.issue(ra, rb, rb, smem, wave, 0);
  int g = 0;   // k-tiles consumed so far: stage g & 1 holds the current one
#pragma unroll 1
  for (; t < last; t += L) {
    const int tn = t + L;
    __amdgpu_buffer_rsrc_t ran = ra, rbn = rb;
    if (tn < last) {
      ran = a_rsrc(tn);
      rbn = b_rsrc(tn);
    }
    const int z = t / tiles, rt = t % tiles, i0 = rt / tpr * kNtTile + wi * 64, j0 = rt % tpr * kNtTile + wj * 128;
    const bool live = i0 < n && j0 < n;   // wave-uniform
    f32x16 acc[4][2];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
      for (int ib = 0; ib < 2; ++ib) acc[jb][ib] = zero16();
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt, ++g) {
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of the k-tile landed
      __syncthreads();                       // ... and everyone's; the other stage is free again
      bf16* nxt = smem + ((g + 1) & 1) * kNtStage;
      if (kt + 1 < nk)
        stg.issue(ra, rb, rb, nxt, wave, (kt + 1) * kNtBK);
      else if (tn < last)
        stg.issue(ran, rbn, rbn, nxt, wave, 0);   // the next tile's first k-tile
      if (live) nt_ktile(smem + (g & 1) * kNtStage, offj, offi, lh, acc);
    }
    // epilogue: plain row-major store of the tile (registers only)
    if (live) {
#pragma unroll
      for (int ib = 0; ib < 2; ++ib) {
        const int i = i0 + ib * 32 + ln;
        bf16* crow = C + z * plane + (size_t)i * ld + j0 + 16 * lh;
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
          float v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = acc[jb][ib][u];
          if (i < n && j0 + jb * 32 + 16 * lh < ld) store16(crow + jb * 32, v);
        }
      }
    }
    ra = ran;
    rb = rbn;
  }
}

// 128 x 128 tiles, one per workgroup.
constexpr int kSmTile = 128;
constexpr int kSmElems = kSmTile * kNtBK;      // one operand tile: [128 rows][8 chunks of 8], chunks swizzled (nt_off)
constexpr int kSmSmem = 2 * 2 * kSmElems * 2;  // bytes: A | B, double-buffered: 64 KB

__global__ __launch_bounds__(256, 2) void bgemm_nt_small_kernel(const bf16* __restrict__ A, const bf16* __restrict__ B,
                                                                bf16* __restrict__ C, int n, int ld, int total) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  bf16* smem = reinterpret_cast<bf16*>(smem_raw);
  const int item = nt_item(total);
  if (item < 0) return;   // the whole workgroup, before any barrier
  const int tpr = (n + kSmTile - 1) / kSmTile, tiles = tpr * tpr;
  const size_t plane = (size_t)n * ld;
  const int z = item / tiles, rt = item % tiles, it = rt / tpr * kSmTile, jt = rt % tpr * kSmTile;
  const int lane = threadIdx.x & 63, wave = wave_id(), ln = lane & 31, lh = lane >> 5;
  const int wi = (wave & 1) * 64, wj = (wave >> 1) * 64;
  const __amdgpu_buffer_rsrc_t ra =
      buffer_rsrc(A + z * plane + (size_t)it * ld, (unsigned)min(n - it, kSmTile) * ld * 2);
  const __amdgpu_buffer_rsrc_t rb =
      buffer_rsrc(B + z * plane + (size_t)jt * ld, (unsigned)min(n - jt, kSmTile) * ld * 2);
  unsigned vo[4];   // wave w copies rows 32 w .. + 31 of each operand, 8 rows (1 KB) at a time
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = wave * 32 + q * 8 + (lane >> 3);
    vo[q] = (unsigned)(row * ld + ((lane & 7) ^ nt_swz(row)) * 8) * 2;
  }
  auto issue = [&](int kt) {
    bf16* st = smem + (kt & 1) * 2 * kSmElems;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      nt_copy16_to_lds(ra, st + (wave * 4 + q) * 512, vo[q], (unsigned)kt * kNtBK * 2);
      nt_copy16_to_lds(rb, st + kSmElems + (wave * 4 + q) * 512, vo[q], (unsigned)kt * kNtBK * 2);
    }
  };
  const bool live = it + wi < n && jt + wj < n;   // wave-uniform
  f32x16 acc[2][2];   // [j block][i block]
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = zero16();
  const int nk = ld / kNtBK;
  issue(0);
#pragma unroll 1
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of the k-tile landed
    __syncthreads();                       // ... and everyone's; the other stage is free again
    if (kt + 1 < nk) issue(kt + 1);
    if (!live) continue;
    const bf16* sa = smem + (kt & 1) * 2 * kSmElems;
    const bf16* sb = sa + kSmElems;
    bf16x8 fi[4][2], fj[4][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        fj[ks][x] = load8(sb + nt_off(wj + x * 32 + perm32(ln), 2 * ks + lh));
        fi[ks][x] = load8(sa + nt_off(wi + x * 32 + ln, 2 * ks + lh));
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = mfma32(fj[ks][x], fi[ks][y], acc[x][y]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!live) return;
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int i = it + wi + y * 32 + ln;
    bf16* crow = C + z * plane + (size_t)i * ld + jt + wj + 16 * lh;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = acc[x][y][u];
      if (i < n && jt + wj + x * 32 + 16 * lh < ld) store16(crow + x * 32, v);
    }
  }
}

// Which tiling: rounds of tiles over the CUs x a round's time in us.  A round of large tiles (one per CU) measured
// 1.9 us per k-tile + 7, one of small tiles (two per CU, half the area) 1.24 + 2.9 (N = 512 and 1024, 128 planes); the
// large kernel's idle waves past n leave it ahead of its estimate, hence the margin.  128 planes, large against small:
// N = 64 4.4 and 4.3 us, 128 6.9 / 6.1, 256 14.0 / 11.3, 333 28.3 / 24.4, 384 29.2 / 26.1 (small), 450 40.2 / 40.9,
// 512 44.5 / 51.1, 773 212 / 228, 1024 299 / 363 (large).  Planes padded to 256 in rows and k took 13.3 us at N = 64,
// 38.9 at 333, 289 at 773.
inline bool use_small_tiles(long long batch, long long n, int cus) {
  const long long t256 = (n + 255) / 256, t128 = (n + 127) / 128;
  const double nk = (double)((n + 63) / 64);
  const double r256 = (double)((batch * t256 * t256 + cus - 1) / cus);
  const double r128 = (double)((batch * t128 * t128 + 2 * cus - 1) / (2 * cus));
  return r128 * (1.24 * nk + 2.9) < 0.85 * r256 * (1.9 * nk + 7.0);
}

}  // namespace

int launch_bgemm_nt(const void* A, const void* B, void* C, int64_t batch, int64_t n, hipStream_t stream) {
  const int64_t ld = bgemm_ld(n);
  const long long tpr = (n + kNtTile - 1) / kNtTile;
  if (n <= 0 || batch <= 0 || batch * 4 * tpr * tpr > (1ll << 31) - 1 || (long long)kNtTile * ld * 2 > 0xffffffffLL) {
    return set_error(BIOEMU_ERR_INVALID_ARG, "bgemm_nt: bad shape batch=%lld n=%lld", (long long)batch,
                     (long long)n);
  }
  int dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
  if (use_small_tiles(batch, n, cus)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(bgemm_nt_small_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kSmSmem) != hipSuccess)
      return set_error(BIOEMU_ERR_LAUNCH, "bgemm_nt: cannot set dynamic LDS size");
    const long long t128 = (n + kSmTile - 1) / kSmTile, total = batch * t128 * t128;
    KernelTimerScope timed("bgemm_nt", stream);
    hipLaunchKernelGGL(bgemm_nt_small_kernel, dim3((unsigned)((total + kNtXcds - 1) / kNtXcds * kNtXcds)), dim3(256),
                       kSmSmem, stream, static_cast<const bf16*>(A), static_cast<const bf16*>(B),
                       static_cast<bf16*>(C), (int)n, (int)ld, (int)total);
    return check_launch("bgemm_nt");
  }
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(bgemm_nt_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          kNtSmem) != hipSuccess)
    return set_error(BIOEMU_ERR_LAUNCH, "bgemm_nt: cannot set dynamic LDS size");
  const long long total = batch * tpr * tpr;
  // one workgroup per CU (128 KB of LDS each), a multiple of the 8 XCDs, no more than the tiles
  const long long nwg = std::max<long long>(kNtXcds, std::min<long long>(cus, (total + kNtXcds - 1) / kNtXcds * kNtXcds)
                                                         / kNtXcds * kNtXcds);
  KernelTimerScope timed("bgemm_nt", stream);
  hipLaunchKernelGGL(bgemm_nt_kernel, dim3((unsigned)nwg), dim3(kNtThreads), kNtSmem, stream,
                     static_cast<const bf16*>(A), static_cast<const bf16*>(B), static_cast<bf16*>(C), (int)n, (int)ld,
                     (int)total, (int)nwg);
  return check_launch("bgemm_nt");
}

}  // namespace bioemu
