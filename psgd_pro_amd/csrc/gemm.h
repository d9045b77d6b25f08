// MFMA products: problems per launch and epilogues, shared by the host launchers and the kernels.
#pragma once
#include "common.h"

namespace psgdk {

constexpr int MAXB = 64;  // problems per grouped launch (pointer arrays in the kernel arguments, by value; the
                          // largest argument block, the norm bound's final stage, is about 8 KB)

// Epilogues. acc is op(A) op(B) accumulated in fp32; s = the problem's device scalars.
enum Epi : int {
  EPI_STORE = 0,   // C = alpha * acc + beta * C
  EPI_FACTOR = 1,  // C = X1 - s[0] * (acc - s[1] * X1)              (Q - lr/L (term1 Q - term2 Q))
  EPI_PROC = 2,    // C = X1 + a X2 + a^2/2 * s[1] * acc, a = s[0]    (Procrustes: Q + a RQ + a^2/2 R RQ)
  EPI_SCALE = 3,   // C = s[0] * acc
  EPI_RQ = 4,      // C = s[0] * acc and trace partials of tr(C), tr(s[0] X1 C) into part[]  (Procrustes RQ)
  EPI_SUMSQ = 5,   // C = alpha * acc and partial sums of C^2 into part[]                    (apply + clip stats)
  EPI_PROCB = 7,   // bf16 kernel only: EPI_PROC with X2 = (R Q)^T in bf16, row stride ldx (the transposed copy
                   // that is also the product's B operand), read at (col, row)
  EPI_STRACE = 6,  // SYRK only: C = (s[0] acc) s[0] (the scale applied twice, so that acc = 0 gives 0 for any
                   // finite s[0]), and partials of sum_ij C_ij X1_ij over the whole symmetric C into part[2 t + 1]
                   // (part[2 t] = 0)                                    (Procrustes r2: S = Rn^T Rn, sum(S * Q))
};

}  // namespace psgdk
