// INT4 group-128 matmul above 16 rows (int4_gemm.hip), called by the Marlin
// entries of int4_marlin.hip.
#pragma once

#include "common.cuh"

// Most rows of one call for this K (0: none; N K / 2 must be below 2^31 too).
__attribute__((visibility("hidden"))) int int4_gemm_rows(int K);

// C[M, N] = A[M, K] @ dequant(W)^T; K % 128 == 0, N % 64 == 0, A 16-byte aligned.
__attribute__((visibility("hidden"))) hipError_t int4_gemm_g128(const f16* A, const uint32_t* Wq, const uint16_t* S,
                                                                const uint32_t* Z, f16* C, int M, int N, int K,
                                                                hipStream_t stream);
