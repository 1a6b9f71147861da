// FP64 matrix-core GEMM entry points (tg_mfma.hip).  `variant` selects the tile of a wave
// (rows x columns, k steps of 4 in flight): 0 = 32x32, 2; 1 = 32x32, 4; 2 = 48x32, 2;
// 3 = 32x48, 2; 4 = 48x32, 3; 5 = 48x16, 3; 6 = 32x16, 3; 7 = 32x16, 4; 8 = 16x16, 2;
// 9 = 16x16, 4; 10 = 48x16, 4.
// Grouped (angles x positions): 0 = 48x32, 2; 1 = 48x32, 3; 2 = 32x32, 4; 3 = 32x32, 2
// (four waves per SIMD); 4 = 16x32, 4; up to TG_GROUPED_VEC angles take matrix-vector
// kernels whatever the variant.
// Batch element b reads A + (b / divA) * sA and B + (b / divB) * sB (an operand shared by
// runs of divA consecutive elements).
#pragma once
#include "tg_internal.h"

constexpr int TG_MFMA_VARIANTS = 11;   // autotuned: 0..10
constexpr int TG_MFMA_GROUPED_VARIANTS = 5;

int mfma_gemm_zz(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const cplx* A, int lda, long long sA, const cplx* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch,
                 int divA = 1, int divB = 1, const GemmEpi& epi = GemmEpi());
int mfma_gemm_dz(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const double* A, int lda, long long sA, const cplx* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch,
                 int divA = 1, int divB = 1, const GemmEpi& epi = GemmEpi());
int mfma_gemm_zd(int variant, hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, cplx alpha,
                 const cplx* A, int lda, long long sA, const double* B, int ldb, long long sB,
                 cplx beta, int use_beta, cplx* C, int ldc, long long sC, int batch,
                 int divA = 1, int divB = 1, const GemmEpi& epi = GemmEpi());
int mfma_gemm_grouped(int variant, hipStream_t s, int M, const cplx* X, cplx* C, int ld,
                      const void* W, const GroupDesc* groups_dev, const int* tile_group_dev,
                      const int* tile_j0_dev, int ntiles_total);
int mfma_gemm_dd(hipStream_t s, TgOp opa, TgOp opb, int M, int N, int K, double alpha,
                 const double* A, int lda, long long sA, const double* B, int ldb, long long sB,
                 double beta, int use_beta, double* C, int ldc, long long sC, int batch,
                 int divA = 1, int divB = 1);
