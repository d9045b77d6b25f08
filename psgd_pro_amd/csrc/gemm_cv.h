// Products of fp32- or bf16-stored operands in any layout, converted while they are staged: argument block shared by
// the host launcher and the kernel.
#pragma once
#include "gemm.h"

namespace psgdk {

// One operand viewed as X[mn][k] (OpMode and sign as in common.h). vec: read 4 consecutive stored elements at a time
// (leading dimension below 2^21; fp32 loads need 4-byte alignment only, bf16 an even row stride and a 4-byte aligned
// base); else element by element.
struct CvOperand {
  int mode, sign, bf16, vec;
  long long ld;
};

// C = epilogue of acc = op(A) op(B) (epilogues of gemm.h; EPI_STORE: alpha acc + beta C).
struct CvArgs {
  int M, N, K;
  CvOperand a, b;
  long long ldc, ldx;
  float alpha, beta;
  int epi;
  int tri;              // 1: upper-triangular tile grid (SYRK: M == N, B is A)
  int gram;             // tri, EPI_STORE, fp32: A may be near a multiple of the identity (64 x 64 tiles keep the diagonal)
  int out_mode;         // tri: 0 upper triangle only, 1 mirrored full matrix, 2 packed upper triangle
  int kbeg;             // 1: A is upper-triangular (A[i][k] = 0 for k < i): a tile's k loop starts at its first row
  int splitk, kchunk;   // split-K (EPI_STORE only): split s covers k in [s kchunk, (s+1) kchunk) and writes its
                        // partial product to C + s * M * ldc
  int f32;              // precision fp32: 1 = fp32 MFMAs instead of three bf16 planes
  int order;            // 0 problem-major tile order, else XCD runs with tile rows grouped by 4
  int tiles_m, tiles_n, ntiles, nb;
  const void* A[MAXB];
  const void* B[MAXB];
  float* C[MAXB];
  const float* X1[MAXB];
  const float* X2[MAXB];
  const float* s[MAXB];
  float* part[MAXB];
};

// Tile configurations: 0 = 128 x 256 (plain rows of one storage type, not A m- with B k-contiguous: gemm_cv_wide), 1 = 64
// x 64, 2 = 32 x 64 (EPI_STORE and EPI_SUMSQ only), 3 = 64 x 64 with k split over two wave groups
bool gemm_cv_wide(const CvArgs& a, int prec);
int gemm_cv_tiles(long long M, long long N, int tri, int cfg);
hipError_t gemm_cv_launch(CvArgs& a, int prec, int cfg, hipStream_t st);

}  // namespace psgdk
