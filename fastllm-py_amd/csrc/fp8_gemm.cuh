// FP8 128x128-block matmul above 16 rows (fp8_gemm.hip), called by the entries
// of fp8.hip.
#pragma once

#include "common.cuh"

#define FP8_GEMM_HIDDEN __attribute__((visibility("hidden")))

// Most rows of one call for this K (0: none; N K must be below 2^31 too).
FP8_GEMM_HIDDEN int fp8_gemm_rows(int K);

// C[M, N] = A[M, K] @ dequant(W)^T (+ bias[N]); K % 64 == 0, K >= 128, A and W
// 16-byte aligned.
FP8_GEMM_HIDDEN hipError_t fp8_gemm_b128(const uint16_t* A, const uint8_t* W, const float* Sc, const uint16_t* bias,
                                         uint16_t* C, int M, int N, int K, bool bf16, hipStream_t stream);
