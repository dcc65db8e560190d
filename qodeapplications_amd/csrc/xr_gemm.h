// Internal GEMM launchers shared by the density and contraction drivers.
#pragma once
#include "xr_common.h"

// FP64 MFMA GEMM (no locking; callers hold the context lock).
// ta = 1: A is K x M (A[k*lda+m]); tb = 1: B is N x K (B[n*ldb+k]).
int xr_dgemm_launch(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                    const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb,
                    int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int64_t batch);

// C = alpha A^T A (A: K x n, C: n x n): upper tiles, then the mirror.
int xr_dgemm_syrk_tn(xr_ctx* c, int64_t n, int64_t K, double alpha, const double* A, int64_t lda, double* C,
                     int64_t ldc);
int xr_dgemm_syrk_nt(xr_ctx* c, int64_t n, int64_t K, double alpha, const double* A, int64_t lda, double* C,
                     int64_t ldc);

// C = A B for A (M x K, M = row[n]) cut into row blocks [row[q], row[q + 1]),
// one grouped launch.  *off == 0 (device): A vanishes outside its diagonal
// blocks, and each row block runs over its own k range only.
int xr_dgemm_blocks(xr_ctx* c, int n, const int64_t* row, int64_t K, int64_t N, const double* A, int64_t lda,
                    const double* B, int64_t ldb, double* C, int64_t ldc, const int* off);

// Split-FP32 product (hi/lo FP32 MFMA, FP64 accumulation) and the
// precision-switched GEMM used by the two-electron contractions.
int xr_dgemm_split_launch(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                          const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb,
                          int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int64_t batch);
// Split-int8 product (Ozaki digit planes on the int8 MFMA).
int xr_dgemm_i8_launch(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                       const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB,
                       double beta, double* C, int64_t ldc, int64_t sC, int64_t batch);
bool xr_i8_pays(int64_t M, int64_t N, int64_t K, int64_t batch);
int xr_gemm_2e(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
               const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB,
               double beta, double* C, int64_t ldc, int64_t sC, int64_t batch);
