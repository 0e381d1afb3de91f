// Host interface of the split-operand GEMMs (split_gemm.hip).
#pragma once

#include "split.h"

namespace bioemu {

constexpr int kSplitStore = 0;     // out = v (+ res)
constexpr int kSplitSwiGLU = 1;    // fc1 / fc2 column blocks interleaved; silu(a) b as operand fragments
constexpr int kSplitQkvg = 2;      // the four token projections of an attention
constexpr int kSplitHidden = 3;    // kSplitStore of kSplitSwiGLU's rows, which have a scale per 32 columns

struct SplitGemmEpi {
  float* out = nullptr;          // kSplitQkvg: q
  const float* bias = nullptr;   // kSplitQkvg: q bias
  const float* res = nullptr;
  int ldo = 0;                   // row length of out (kSplitQkvg: c_s)
  float *k = nullptr, *v = nullptr, *g = nullptr;   // kSplitQkvg
  int T = 0;                                        // kSplitQkvg: v transposed per sequence of T rows (0: row-major)
  f16* hfrag = nullptr;          // kSplitSwiGLU: [row block][hsteps] fragments, and 1 / scale [hidden / 32][M]
  float* hinv = nullptr;
  int hsteps = 0;
};

// Widest row split_prep holds in registers (12 k-steps in each of 4 waves); longer rows are read once per pass.
constexpr int kSplitMaxK = 12 * 4 * 16;
// Fewest 128 x 128 tiles worth the tiled kernel.
constexpr int kSplitTiledMin = 128;

// M rows x N columns (N % 32 == 0; kSplitSwiGLU: both matrices' columns), K columns of A and W fragments (kSplitHidden:
// K % 32 == 0, ainv of kSplitSwiGLU).
int split_gemm(int epi, const f16* A, const float* ainv, const f16* W, const float* winv, const SplitGemmEpi& e,
               long long M, int K, int N, hipStream_t stream, const char* name);

// The same straight from M fp32 rows of 128 channels; kSplitStore and kSplitQkvg.  With wbias (kSplitQkvg) the rows
// are LayerNormed, the affine folded into W and wbias (SplitMat).
int split_gemm_r128(int epi, const float* x, const f16* W, const float* winv, const float* wbias,
                    const SplitGemmEpi& e, long long M, int N, hipStream_t stream, const char* name);

}  // namespace bioemu
