// The product for 17 to 64 rows that finishes in one launch (gemm_rows_bf16.hip), called from the tiled product's launch code.
#pragma once
#include "common.h"

constexpr int GEMM_ROWS_MAX = 64;
constexpr int GEMM_ROWS_MIN_K = 1024;  // two steps of 64 columns for each of a block's waves

// What goes with a norm folded into the product.  A product that reads a row which another left for the norm: ss
// [M][parts] sums of x^2, eps; g null.  A product into the residual that leaves such a row: g the norm's weight [N], raw
// [M][ld_raw] takes bfloat16(x g), ss [M][parts = N / 16] the sums of x^2 of every band.  act: the activation of mode 5.
struct RowsNorm {
  float* ss = nullptr;
  int parts = 0;
  float eps = 0.f;
  const float* g = nullptr;
  bf16_t* raw = nullptr;
  int ld_raw = 0;
  int act = 0;
};
// q, k and v (heads in this order, whole heads rotated, pairs (e, e + d/2)): see gemm_bf16.hip's FinishRope
struct RowsRope {
  const float* cos_sin = nullptr;
  const int* positions = nullptr;
  const int* row_seg = nullptr;
  const int* block_table = nullptr;
  int max_blocks = 0;
  bf16_t* cache = nullptr;
  int P = 0, H = 0, Hk = 0, d = 0;
};

// mode: 0 store bfloat16, 1 store float32, 2 add into float32, 3 SwiGLU (W = gate, W2 = up, N = the width of each), 5 an
// activation, stored in bfloat16.  W, W2 in the tiled layout.
bool gemm_rows_takes(int mode, const void* A, int lda, const void* W, const void* W2, const void* C, int ldc, int M, int N, int K);
int launch_gemm_rows(int mode, const bf16_t* A, int lda, const bf16_t* W, const bf16_t* W2, void* C, int ldc, int M, int N, int K,
                     const RowsNorm& norm, hipStream_t stream);
bool gemm_rows_qkv_takes(const void* A, int lda, const void* W, const void* q_out, int ldq, int M, int K, int H, int Hk, int d,
                         const void* cos_sin, const void* cache);
int launch_gemm_rows_qkv(const bf16_t* A, int lda, const bf16_t* W, bf16_t* q_out, int ldq, int M, int K, const RowsNorm& norm,
                         const RowsRope& rope, hipStream_t stream);
