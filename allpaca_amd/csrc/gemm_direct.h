// The product for many rows that loads its weights straight into registers (gemm_direct_bf16.hip), called from the
// tiled product's launch code.
#pragma once
#include "common.h"

// From so many rows on whatever the columns.
constexpr int GEMM_DIRECT_MIN_ROWS = 1024;
// Fewer rows, K in one piece: where the 128 x 128 tile (64 outputs wide for SwiGLU) would not get by with one tile a
// compute unit.  Microseconds, that tile / this kernel, K 4,096: 768 rows x 6,144 outputs (288 tiles) 63 / 50, 1,000 x
// 4,096 (256 tiles) 43 / 48, 512 x 6,144 (192) 42 / 49; K 3,072: 896 x 5,120 (280) 49 / 38, 768 x 5,120 (240) 34 / 38;
// SwiGLU of 14,336 outputs, K 4,096: 128 rows (224) 53 / 67, 130 (448) 75 / 59, 256 (448) 79 / 67; of 8,192 outputs, K 3,072:
// 256 rows (256) 37 / 48, 384 (384) 54 / 49.
constexpr int GEMM_DIRECT_FEW_ROWS = 129;

// mode: 0 store bfloat16, 1 store float32, 2 add into float32, 3 SwiGLU (W = gate, W2 = up, N = the width of each).
// True if launch_gemm_direct runs this shape (K a multiple of 128, N and ldc of 4, 16-byte aligned A and C, ...).
bool gemm_direct_takes(int mode, const void* A, int lda, const void* C, int ldc, int M, int N, int K);
// W, W2 in the tiled layout.  APC_ERR_UNSUPPORTED for a shape that gemm_direct_takes refuses.
int launch_gemm_direct(int mode, const bf16_t* A, int lda, const bf16_t* W, const bf16_t* W2, void* C, int ldc, int M,
                       int N, int K, hipStream_t stream);
// Mode 0 with an activation (see activation_f) on the sums; for shapes that gemm_direct_takes in mode 0.
int launch_gemm_direct_act(int act, const bf16_t* A, int lda, const bf16_t* W, void* C, int ldc, int M, int N, int K,
                           hipStream_t stream);
// Products on rows that a product into the residual left for the RMS norm (A = the rows times the norm's weight, ss =
// [M][ss_parts] sums of x^2): the sums are scaled by 1 / sqrt(sum(ss[m]) / K + eps), before the activation where there
// is one.  mode 0 (store bfloat16) or 3 (SwiGLU).
bool gemm_direct_pre_takes(int mode, const void* A, int lda, const void* C, int ldc, int M, int N, int K, int ss_parts);
int launch_gemm_direct_pre(int mode, const bf16_t* A, int lda, const float* ss, int ss_parts, float eps, const bf16_t* W,
                           const bf16_t* W2, void* C, int ldc, int M, int N, int K, hipStream_t stream);
// The product into the float32 residual C that also leaves the row for the RMS norm that reads the residual next:
// raw [M][ldr] = bfloat16(C g) and ss [M][parts] = sums of C^2 over parts of the columns.  gemm_direct_emit_parts says
// how many parts these sizes give (0: not taken; which depends on whether K goes in slices and on the tiles chosen);
// workspace: room for gemm_direct_emit_k_split(M, N, K) * M * N floats where that is more than 1.
int gemm_direct_emit_parts(const void* A, int lda, const void* C, int ldc, int M, int N, int K);
int launch_gemm_direct_emit(const bf16_t* A, int lda, const bf16_t* W, float* C, int ldc, int M, int N, int K,
                            const float* g, bf16_t* raw, int ldr, float* ss, int ss_parts, float* workspace,
                            hipStream_t stream);
// Slices of K that a product of M rows into N columns should be cut into (1: none).  With more than one:
// launch_gemm_direct_slices leaves float32 sums in partials[slice][M][N], K a multiple of k_split * 128.
int gemm_direct_k_split(int M, int N, int K);
int gemm_direct_emit_k_split(int M, int N, int K);   // of launch_gemm_direct_emit
int launch_gemm_direct_slices(const bf16_t* A, int lda, const bf16_t* W, float* partials, int M, int N, int K,
                              int k_split, hipStream_t stream);
