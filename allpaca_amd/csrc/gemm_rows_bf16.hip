// Matrix product for 17 to 64 rows (a decode step of many requests):  C[M,N] = A[M,K] . W[N,K]^T, bfloat16 in, float32
// sums, finished in one launch.
//
// As in skinny_gemm_bf16.hip the weights (tiles of 16 rows x 32 columns in operand order) go from memory straight into
// MFMA operands, each read once by one wave, and a block's eight waves take an eighth of K each and meet in LDS, so no sums
// go through memory and no second kernel adds them.  What is new with more rows is the activations: every block reads all
// M x K of them, and they come out of L2 at 131 GB/s a compute unit in whole lines of 128 bytes.  That is why a block takes
// up to four bands of 16 outputs where there are bands enough.
//  * A step is 64 columns of K: of NB bands two tiles each, and of every 16 rows two loads of 8 rows x 128 bytes, eight
//    lanes side by side a line.  (Loads whose lanes sit where the operands want them, eight rows in eight lanes, come at
//    35 GB/s a compute unit: 64 rows x 4,096 columns of K into 4,096 outputs 20.4 us, so 14.4.)  They go
//    through the wave's own part of LDS, eight pieces of 16 bytes a row in an order that depends on the row, to the lanes
//    that want them; a wave's LDS accesses are served in order, so there is no barrier in the loop.
//  * DEPTH register sets of a step: what a compute unit has in flight is 8 waves x DEPTH x NB x 2 KiB of weights.
//  * Operands as in skinny_gemm_bf16.hip (weights first): a lane ends with four consecutive outputs of a row.
// Bound by a fixed part of some 5 us (first loads, the waves' meeting, the store) and the activations' way: with the weights
// beside them a compute unit gets 33-60 GB/s in all.  Times, and where the tiled kernel is the better one: gemm_rows_takes.
// K must be a multiple of 64, from 1,024 on; N of 16.
// The order of additions for an output depends on K alone.
// Reference counterpart: gemm_nt_bf16_tiled_kernel, hip/src/kernels.cpp:634 (no matrix cores there).
#include "gemm_rows.h"
#include "host/rules.h"
#include "mfma.h"

namespace {

enum { R_STORE_BF16 = 0, R_STORE_F32 = 1, R_ACC_F32 = 2, R_SWIGLU = 3, R_QKV_ROPE = 4, R_ACT = 5 };
constexpr int WAVES = 8;
constexpr int TILE_ELEMS = 16 * 32;
// outputs' bands of a block that hold NB bands of weights
__host__ __device__ constexpr int out_bands(int mode, int nb) { return mode == R_SWIGLU ? nb / 2 : mode == R_QKV_ROPE ? 1 : nb; }
// register sets of a step, NB x 8 registers of weights and MT x 8 of activations each (one or two more are slower: 64 rows
// x 4,096 columns of K into 4,096 outputs 14.4 us with 3 sets, 18 with 5)
constexpr int depth_of(int mt, int nb) { return nb == 4 ? 2 : nb == 1 && mt < 4 ? 4 : 3; }

template <int MT, int NB>
struct RowsSet {
  Frag w[NB][2];
  Frag a[MT][2];
};

template <int MT, int NB, int MODE, bool PRE, bool EMIT>
__global__ __launch_bounds__(WAVES * 64, 1) void rows_gemm_kernel(const bf16_t* __restrict__ A, int lda,
                                                                 const bf16_t* __restrict__ W,
                                                                 const bf16_t* __restrict__ W2, int chunks,
                                                                 void* __restrict__ C, int ldc, int M, int N, int K,
                                                                 RowsNorm norm, RowsRope rope) {
  static_assert(MODE != R_QKV_ROPE || NB == 2, "the two bands of a block hold the two halves of the pairs");
  static_assert(!EMIT || MODE == R_ACC_F32, "only a product that adds into the residual leaves the next norm's row");
  constexpr int OUT = out_bands(MODE, NB), SUMS = NB / OUT, DEPTH = depth_of(MT, NB);
  // a wave's activations of a step on their way to the operands, in the end its sums
  constexpr int PART = (NB > 2 ? NB : 2) * MT * 1024;
  __shared__ __attribute__((aligned(1024))) unsigned char part[WAVES][PART];
  __shared__ float rstd_s[PRE ? MT * 16 : 1];
  const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int i = lane % 16, c = lane / 16;
  const int bands = N / 16, band0 = blockIdx.x * OUT;

  // bands of weights: SwiGLU the OUT gate bands, then the same bands of up; q, k, v the bands j and j + d / 32 of a head
  const bf16_t* wb[NB];
  const int head = MODE == R_QKV_ROPE ? (int)blockIdx.x / (rope.d / 32) : 0, head_band = MODE == R_QKV_ROPE ? (int)blockIdx.x % (rope.d / 32) : 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int band = MODE == R_QKV_ROPE ? head * (rope.d / 16) + head_band + b * (rope.d / 32) : min(band0 + b % OUT, bands - 1);
    wb[b] = (MODE == R_SWIGLU && b >= OUT ? W2 : W) + (size_t)band * chunks * TILE_ELEMS + lane * 8;
  }
  // loads of 8 rows x 128 bytes: lane -> (row lane / 8, 16 bytes lane % 8), in LDS at 16 bytes lane % 8 ^ row; read back row i,
  // 16 bytes c (a step's first tile) or 4 + c (its second)
  uint32_t arow[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      arow[t][h] = (uint32_t)min(t * 16 + h * 8 + lane / 8, M - 1) * (uint32_t)lda + (lane % 8) * 8;
  unsigned char* mine = &part[wave][0];
  const int put = (lane / 8) * 128 + ((lane % 8) ^ (lane / 8)) * 16;
  const int get0 = i * 128 + ((c ^ (i % 8)) * 16), get1 = i * 128 + (((4 + c) ^ (i % 8)) * 16);

  floatx4 acc[NB][MT];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[b][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto load_step = [&](RowsSet<MT, NB>& r, int s) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 2; ++u) r.w[b][u] = load_frag_once(wb[b] + (size_t)(2 * s + u) * TILE_ELEMS);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) r.a[t][h] = load_frag(A + s * 64 + arow[t][h]);
  };
  auto compute = [&](const RowsSet<MT, NB>& r) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<Frag*>(mine + (t * 2 + h) * 1024 + put) = r.a[t][h];
    wave_lds_order();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const Frag first = *reinterpret_cast<const Frag*>(mine + t * 2048 + get0);
      const Frag second = *reinterpret_cast<const Frag*>(mine + t * 2048 + get1);
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b][t] = mfma16(r.w[b][0], first, acc[b][t]);
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b][t] = mfma16(r.w[b][1], second, acc[b][t]);
    }
    wave_lds_order();
  };

  // this wave's steps, at least two (GEMM_ROWS_MIN_K); DEPTH loaded ahead, no branch around a load in the loop
  const int steps = K / 64, lo = wave * steps / WAVES, n = (wave + 1) * steps / WAVES - lo, last = lo + n - 1;
  // All blocks walk K in the same order: a SwiGLU whose blocks begin at different steps of a wave's range asks L2 for fewer equal
  // lines at a time (64 rows, K 3,072 into 8,192 outputs 23.5 us in step, 22.3 so), but adds an output in its own order a block
  RowsSet<MT, NB> set[DEPTH];
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load_step(set[d], min(lo + d, last));

  // Behind the first loads: the rows' scale (8 threads a row), and what the finishing waves add to or rotate by
  if constexpr (PRE) {
#pragma unroll
    for (int m0 = 0; m0 < MT * 16; m0 += WAVES * 8) {
      const int m = m0 + tid / 8;
      const float sum = row_parts_sum<8>(norm.ss + (size_t)min(m, M - 1) * norm.parts, norm.parts, tid % 8);
      if (tid % 8 == 0 && m < MT * 16) rstd_s[m] = 1.0f / sqrtf(sum / (float)K + norm.eps);
    }
  }
  constexpr int ITEMS = OUT * MT, ROUNDS = (ITEMS + WAVES - 1) / WAVES;  // (band, 16 rows) to finish, dealt out to the waves
  // (64 rows and four bands leave no registers for the norm's weight: it is asked for at the end)
  constexpr bool G_EARLY = MT * NB < 16;
  floatx4 old[ROUNDS], gv[ROUNDS];
  if constexpr (MODE == R_ACC_F32) {
#pragma unroll
    for (int q = 0; q < ROUNDS; ++q) {
      const int item = q * WAVES + wave, m = item % MT * 16 + i, nn = (band0 + item / MT) * 16 + c * 4;
      old[q] = gv[q] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (item < ITEMS && m < M && nn < N) {
        old[q] = *reinterpret_cast<const floatx4*>((const float*)C + (size_t)m * ldc + nn);
        if constexpr (EMIT && G_EARLY) gv[q] = *reinterpret_cast<const floatx4*>(norm.g + nn);
      }
    }
  }
  floatx4 cosv = floatx4{0.f, 0.f, 0.f, 0.f}, sinv = floatx4{0.f, 0.f, 0.f, 0.f};
  int pos = 0, page_id = 0;
  const int e0 = head_band * 16 + c * 4;  // q, k, v: this lane's first element of the head's first half
  if constexpr (MODE == R_QKV_ROPE) {
    const int m = wave * 16 + i;
    if (wave < MT && m < M) {
      pos = rope.positions[m];
      const float* cs = rope.cos_sin + (size_t)pos * rope.d + e0;
      cosv = *reinterpret_cast<const floatx4*>(cs);
      sinv = *reinterpret_cast<const floatx4*>(cs + rope.d / 2);
      if (head >= rope.H) page_id = rope.block_table[(size_t)rope.row_seg[m] * rope.max_blocks + pos / rope.P];
    }
  }

  int t = 0;
  for (; t + DEPTH < n; t += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      compute(set[d]);
      load_step(set[d], min(lo + t + d + DEPTH, last));
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (t + d < n) compute(set[d]);

  // the waves' sums, added in wave order
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < MT; ++r) *reinterpret_cast<floatx4*>(mine + ((b * MT + r) * 64 + lane) * 16) = acc[b][r];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < ROUNDS; ++q) {
    const int item = q * WAVES + wave;
    if (item >= ITEMS) break;
    const int b = item / MT, rt = item % MT, m = rt * 16 + i;
    floatx4 sum[SUMS];
#pragma unroll
    for (int s = 0; s < SUMS; ++s) {
      sum[s] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) sum[s] += *reinterpret_cast<const floatx4*>(&part[w][(((b + s * OUT) * MT + rt) * 64 + lane) * 16]);
      if constexpr (PRE) sum[s] *= rstd_s[m];
    }
    if constexpr (MODE == R_QKV_ROPE) {
      if (m >= M) continue;
      bf16_t* page = rope.cache + (size_t)page_id * ((size_t)2 * rope.Hk * rope.P * rope.d);
      const int half = rope.d / 2, slot = pos % rope.P;
      if (head >= rope.H + rope.Hk) {
        bf16_t* col = page + (size_t)rope.Hk * rope.P * rope.d + ((size_t)(head - rope.H - rope.Hk) * rope.d + e0) * rope.P + slot;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          col[(size_t)r * rope.P] = float_to_bf16(sum[0][r]);
          col[(size_t)(half + r) * rope.P] = float_to_bf16(sum[SUMS - 1][r]);
        }
        continue;
      }
      float ya[4], yb[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float av = bf16_to_float(float_to_bf16(sum[0][r])), bv = bf16_to_float(float_to_bf16(sum[SUMS - 1][r]));
        ya[r] = av * cosv[r] - bv * sinv[r];
        yb[r] = av * sinv[r] + bv * cosv[r];
      }
      bf16_t* dst = head < rope.H ? (bf16_t*)C + (size_t)m * ldc + (size_t)head * rope.d
                                  : page + ((size_t)(head - rope.H) * rope.P + slot) * rope.d;
      *reinterpret_cast<uint2*>(dst + e0) = uint2{pack_bf16x2(ya[0], ya[1]), pack_bf16x2(ya[2], ya[3])};
      *reinterpret_cast<uint2*>(dst + e0 + half) = uint2{pack_bf16x2(yb[0], yb[1]), pack_bf16x2(yb[2], yb[3])};
      continue;
    }
    const int nn = (band0 + b) * 16 + c * 4;
    const bool on = m < M && nn < N;
    if constexpr (MODE == R_ACC_F32) {
      const floatx4 x = old[q] + sum[0];
      if constexpr (EMIT && !G_EARLY) {
        if (on) gv[q] = *reinterpret_cast<const floatx4*>(norm.g + nn);
      }
      if (on) *reinterpret_cast<floatx4*>((float*)C + (size_t)m * ldc + nn) = x;
      if constexpr (EMIT) {
        if (on)
          *reinterpret_cast<uint2*>(norm.raw + (size_t)m * norm.ld_raw + nn) =
              uint2{pack_bf16x2(x[0] * gv[q][0], x[1] * gv[q][1]), pack_bf16x2(x[2] * gv[q][2], x[3] * gv[q][3])};
        float sq = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
        sq += __shfl_xor(sq, 16, WAVE);  // the four lanes with pieces of the row
        sq += __shfl_xor(sq, 32, WAVE);
        if (c == 0 && on) norm.ss[(size_t)m * norm.parts + band0 + b] = sq;
      }
    } else if (on) {
      if constexpr (MODE == R_STORE_F32) {
        *reinterpret_cast<floatx4*>((float*)C + (size_t)m * ldc + nn) = sum[0];
      } else {
        floatx4 y = sum[0];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (MODE == R_SWIGLU) y[r] = silu_f(sum[0][r]) * sum[SUMS - 1][r];
          if (MODE == R_ACT) y[r] = activation_f(sum[0][r], norm.act);
        }
        *reinterpret_cast<uint2*>((bf16_t*)C + (size_t)m * ldc + nn) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      }
    }
  }
}

int kind_of(int mode) {
  return mode == R_SWIGLU ? apc_rules::ROWS_GATED : mode == R_QKV_ROPE ? apc_rules::ROWS_QKV : apc_rules::ROWS_PLAIN;
}

template <int MODE, bool PRE, bool EMIT>
int launch(const bf16_t* A, int lda, const bf16_t* W, const bf16_t* W2, void* C, int ldc, int M, int N, int K, RowsNorm norm,
           RowsRope rope, hipStream_t stream) {
  const int bands = N / 16, mt = ceil_div(M, 16);
#define ROWS_LAUNCH(MT_, NB_, BLOCKS_)                                                                             \
  hipLaunchKernelGGL((rows_gemm_kernel<MT_, NB_, MODE, PRE, EMIT>), dim3(BLOCKS_), dim3(WAVES * 64), 0, stream, A, lda, \
                     W, W2, ceil_div(K, 32), C, ldc, M, N, K, norm, rope)
#define ROWS_BY_M(NB_, BLOCKS_)                \
  if (mt == 2) ROWS_LAUNCH(2, NB_, BLOCKS_);   \
  else if (mt == 3) ROWS_LAUNCH(3, NB_, BLOCKS_); \
  else ROWS_LAUNCH(4, NB_, BLOCKS_)
  if constexpr (MODE == R_QKV_ROPE) {
    ROWS_BY_M(2, bands / 2);
  } else {
    const int nb = apc_rules::rows_bands(M, N, K, kind_of(MODE));
    if (nb == 4) { ROWS_BY_M(4, ceil_div(bands, out_bands(MODE, 4))); }
    else if (nb == 2) { ROWS_BY_M(2, ceil_div(bands, out_bands(MODE, 2))); }
    else if constexpr (MODE != R_SWIGLU) { ROWS_BY_M(1, bands); }
  }
#undef ROWS_BY_M
#undef ROWS_LAUNCH
  APC_LAUNCH_CHECK();
  return 0;
}

bool aligned(const void* p, unsigned n) { return ((uintptr_t)p & (n - 1)) == 0; }
}  // namespace

// Where the tiled kernel is the better one: apc_rules::rows_bands.  Microseconds in a step of 64 rows at 3B shapes, tiled kernel
// and adding kernel / this: q, k, v with rotation and cache 18.9 / 16.8, o_proj with the norm's row 14.4 / 12.2, SwiGLU of
// 8,192 27.1 / 23.7.  In a loop: 32 rows, K 2,048 into 3,072 outputs 13 / 6.1, K 4,096 into 4,096 16.6 / 10.7; 64 rows, K 4,096
// into 4,096 17.7 / 14.2; the other way: 64 rows, K 8,192 into 3,072 18.4 / 23.6, 32 rows, K 14,336 into 4,096 27.4 / 32.9.
bool gemm_rows_takes(int mode, const void* A, int lda, const void* W, const void* W2, const void* C, int ldc, int M, int N, int K) {
  const bool out32 = mode == R_STORE_F32 || mode == R_ACC_F32;
  if (M <= 16 || M > GEMM_ROWS_MAX || K < GEMM_ROWS_MIN_K || K % 64 || N <= 0 || N % 16 || lda % 8 || lda >= (1 << 24) || ldc % 4 ||
      !aligned(A, 16) || !aligned(W, 16) || !aligned(W2, 16) || !aligned(C, out32 ? 16 : 8))
    return false;
  return apc_rules::rows_bands(M, N, K, kind_of(mode)) > 0;
}

int launch_gemm_rows(int mode, const bf16_t* A, int lda, const bf16_t* W, const bf16_t* W2, void* C, int ldc, int M, int N, int K,
                     const RowsNorm& norm, hipStream_t stream) {
  if (!gemm_rows_takes(mode, A, lda, W, W2, C, ldc, M, N, K)) return APC_ERR_UNSUPPORTED;
  const RowsRope none{};
  const bool pre = norm.ss && !norm.g;
#define ROWS(MODE_, PRE_) return launch<MODE_, PRE_, false>(A, lda, W, W2, C, ldc, M, N, K, norm, none, stream)
  switch (mode) {
    case R_STORE_BF16: if (pre) ROWS(R_STORE_BF16, true); ROWS(R_STORE_BF16, false);
    case R_STORE_F32: if (pre) ROWS(R_STORE_F32, true); ROWS(R_STORE_F32, false);
    case R_SWIGLU: if (pre) ROWS(R_SWIGLU, true); ROWS(R_SWIGLU, false);
    case R_ACT: if (pre) return APC_ERR_UNSUPPORTED; ROWS(R_ACT, false);
    case R_ACC_F32:
      if (pre) return APC_ERR_UNSUPPORTED;
      if (!norm.g) ROWS(R_ACC_F32, false);
      if (norm.parts != N / 16 || norm.ld_raw % 4 || !aligned(norm.raw, 8) || !aligned(norm.g, 16)) return APC_ERR_UNSUPPORTED;
      return launch<R_ACC_F32, false, true>(A, lda, W, W2, C, ldc, M, N, K, norm, none, stream);
    default: return APC_ERR_BAD_ARG;
  }
#undef ROWS
}

bool gemm_rows_qkv_takes(const void* A, int lda, const void* W, const void* q_out, int ldq, int M, int K, int H, int Hk, int d,
                         const void* cos_sin, const void* cache) {
  return d % 32 == 0 && aligned(cos_sin, 16) && aligned(cache, 8) &&
         gemm_rows_takes(R_QKV_ROPE, A, lda, W, nullptr, q_out, ldq, M, (H + 2 * Hk) * d, K);
}

int launch_gemm_rows_qkv(const bf16_t* A, int lda, const bf16_t* W, bf16_t* q_out, int ldq, int M, int K, const RowsNorm& norm,
                         const RowsRope& rope, hipStream_t stream) {
  if (!gemm_rows_qkv_takes(A, lda, W, q_out, ldq, M, K, rope.H, rope.Hk, rope.d, rope.cos_sin, rope.cache)) return APC_ERR_UNSUPPORTED;
  const int N = (rope.H + 2 * rope.Hk) * rope.d;
  if (norm.ss) return launch<R_QKV_ROPE, true, false>(A, lda, W, nullptr, q_out, ldq, M, N, K, norm, rope, stream);
  return launch<R_QKV_ROPE, false, false>(A, lda, W, nullptr, q_out, ldq, M, N, K, norm, rope, stream);
}
