// The quantised GEMM of 9 to 64 rows (qmm_short.hip).
#pragma once
#include "common.h"

// Inputs that it can take: kQmmShortMinRows (fewer: the GEMV family) to kQmmShortMaxRows rows, K of whole groups
// whose scales fit beside the activations in LDS.  9 to 16 rows are those of 8-bit models, which leave the GEMVs
// at 8: pair of 14336x4096 under 12 rows 35 us (128-row tile 55, two products that split K and the SwiGLU 49),
// of 8192x2048 13 (20, 27); 4096x14336 20.7 (25), 6144x4096 12.8 (16.5).
// (two blocks of 64 rows would read the weights twice: pair of 14336x4096 under 126 rows 61 us against 54)
constexpr int kQmmShortMinRows = 9, kQmmShortMaxRows = 64;
constexpr int kQmmShortMaxK = 32768;
inline bool exo_qmm_short_can(int M, int K) {
  return M >= kQmmShortMinRows && M <= kQmmShortMaxRows && K % 64 == 0 && K <= kQmmShortMaxK;
}

// whether the pair is faster here than on the 128-row tile.  A product without room to split K answers alike,
// so that the pair keeps the bits of two such products.
bool exo_qmm_short_fits(int M, int N, int K, int bits);

// parts of K that a launch without a second matrix is best split into, where it has room for their sums
int exo_qmm_short_parts(int M, int N, int K);

// whether such a launch is faster than the tiles that split K over workgroups (qmm.hip), where those can be had
bool exo_qmm_short_beats_split(int M, int N, int K);

// y[M,N] = x w^T (+ residual), or with a second matrix silu(x w^T) * (x w2^T); with several parts of K only their
// float32 sums, to part[parts][part_stride]
void exo_qmm_short(const bf16_t* x, const uint32_t* w, const bf16_t* s, const bf16_t* b, const uint32_t* w2,
                   const bf16_t* s2, const bf16_t* b2, const bf16_t* residual, bf16_t* y, int M, int N, int K, int bits,
                   int parts, float* part, size_t part_stride, hipStream_t stream);
