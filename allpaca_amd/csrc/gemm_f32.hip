// Matrix product  C[M,N] = A[M,K] . W[N,K]^T  of float32 operands on the matrix cores (v_mfma_f32_16x16x4_f32: float32
// products and sums, no reduced mode).
//
// Every output is  s0 + s1 + .. + s7  added in this order; slice i is the chain over k in [i L, (i+1) L), L the
// multiple of 32 that eight of cover K, four k an instruction, sixteen k in the order 0 4 8 12, 1 5 9 13, .. .  That
// depends on K alone, not on M, N, the tile or the grid: a row of a batch equals that row computed alone bit for bit.
//
// The eight slices are the eight waves of a block.  Each computes the block's whole tile over its own k and meets the
// others in LDS at the end, so a product with few tiles (decoded rows; 2,048 outputs and a few hundred rows) still has
// eight waves a compute unit at work, no wave waits for another inside the loop, and there are no partial sums in
// memory.  A wave brings 32 k of its rows into registers as eight lanes a row (128 consecutive bytes; the instruction's
// own operand order would have every lane in another row), D of such stages ahead, and turns them into operands in a
// piece of LDS of its own.
//
// What bounds it: with few rows the bytes of W, else the matrix cores' float32 rate (157 TFLOP/s, of which a library
// product of 8,192^3 reaches 151 and a loop of these instructions 156).  Blocks of the large tiles go on to further tiles
// with the next one's first loads on their way while the eight waves meet, and a stage's LDS stores and loads stand between
// its first half's products: 325 rows x 8,192 outputs of SwiGLU 202 -> 186 us, x 2,048 outputs x K 2,048 32.0 -> 30.6, K
// 8,192 104 -> 99 (110 TFLOP/s).  What is left there: the loads (without them, timing only, 14 % less: their way into the
// registers beside the products) and, for every tile, 3 us in which the waves meet.  Measured, microseconds (in brackets
// the kernel of one fma chain an output on the vector units, which takes the other types): 4 rows x 2,048 outputs x K
// 2,048 6.7; x 128,256 outputs 151 (7.0 TB/s); 325 rows x 8,192 outputs of SwiGLU 186 (about 1,600; 117 TFLOP/s); 2,048
// rows x 2,048 outputs x K 8,192 512 (134 TFLOP/s).  All times in this file: launches of a graph one behind the other, weights
// that no launch has just read; inside a step the same products take up to 1 us more.
#include "mfma.h"
#include <math.h>

namespace {

constexpr int SLICES = 8, STAGE = 32;
constexpr int NORM_K = 4096;            // the longest row that a product normalises by itself

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool ONCE>
__device__ __forceinline__ f32x4 load_f32x4(BufferRsrc rsrc, int lane_bytes, int scalar_bytes) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(f32x4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_bytes, scalar_bytes, ONCE ? 2 : 0));
}
template <int N>
struct Count { static constexpr int value = N; };
template <int N, typename F>
__device__ __forceinline__ void each_count(F f) {        // f(1), .. f(N), known when compiling
  if constexpr (N > 1) each_count<N - 1>(f);
  f(Count<N>{});
}

__device__ __forceinline__ float row_scale(float squares, int K, float eps) { return 1.0f / sqrtf(squares / (float)K + eps); }

// H = A * G and R = 1 / sqrt(mean square + eps) of rows in front of an RMS norm, with the operations of the product's NORMALISED
// form and in its order: the squares of a slice's k are added by four chains, one a quarter of every 16 k, as an operand's lanes
// hold them there.  Two forms of the same bits.  Here the 32 lanes that add read the row themselves, two rows a wave: for rows so
// many that they fill the chip, and short ones.
__global__ __launch_bounds__(64) void norm_rows_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ G, float eps,
                                                           float* __restrict__ H, float* __restrict__ R, int M, int K) {
  const int lane = threadIdx.x % 32, m = min((int)(blockIdx.x * 2 + threadIdx.x / 32), M - 1);   // (a last row twice: the same values)
  const int slice = STAGE * ((K + STAGE * SLICES - 1) / (STAGE * SLICES)), k0 = lane / 4 * slice, end = min(K, k0 + slice);
  const float* a = A + (size_t)m * lda;
  float ss[2] = {0.f, 0.f};
  for (int k = k0 + lane % 4 * 4; k < end; k += 128) {
    f32x4 v[8], g[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = g[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + 16 * u < end) v[u] = *(const f32x4*)(a + k + 16 * u), g[u] = *(const f32x4*)(G + k + 16 * u);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) ss[e % 2] = fmaf(v[u][e], v[u][e], ss[e % 2]), v[u][e] *= g[u][e];
      if (k + 16 * u < end) *(f32x4*)(H + (size_t)m * K + k + 16 * u) = v[u];
    }
  }
  float own = ss[0] + ss[1];
  own += __shfl_xor(own, 1), own += __shfl_xor(own, 2);
  float all = 0.f;
#pragma unroll
  for (int w = 0; w < SLICES; ++w) all += __shfl(own, w * 4, 32);
  if (lane == 0) R[m] = row_scale(all, K, eps);
}

// Here a block takes a row: every thread has pieces of the eight slices, and they go through LDS to the 32 lanes of the first wave
// that add.  Bound by the row's way: 32 lanes have an eighth of a long row's loads in flight at a time.
constexpr int NORM_PASSES = 4, NORM_PITCH = 36;         // passes of 128 k of every slice; 16-byte pieces between slices (banks)
__global__ __launch_bounds__(256) void norm_row_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ G, float eps,
                                                            float* __restrict__ H, float* __restrict__ R, int M, int K) {
  extern __shared__ f32x4 room[];                       // [group % 2][pass][slice][piece], what K needs of it
  const int m = blockIdx.x, own = threadIdx.x / 32, at = threadIdx.x % 32;     // this thread's slice, its piece of a pass of it
  const int slice = STAGE * ((K + STAGE * SLICES - 1) / (STAGE * SLICES));
  const int passes = (slice + 127) / 128, groups = (passes + NORM_PASSES - 1) / NORM_PASSES;
  const float* a = A + (size_t)m * lda;
  f32x4 v[NORM_PASSES], g[NORM_PASSES];
  auto column = [&](int group, int u, bool& in) __attribute__((always_inline)) {
    const int o = (group * NORM_PASSES + u) * 128 + at * 4, k = own * slice + o;
    in = o < slice && k < K;
    return in ? k : 0;
  };
  auto load = [&](int group) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NORM_PASSES; ++u) {
      bool in;
      const int k = column(group, u, in);
      v[u] = *(const f32x4*)(a + k), g[u] = *(const f32x4*)(G + k);
    }
  };
  load(0);
  float ss[2] = {0.f, 0.f};
  for (int group = 0; group < groups; ++group) {
#pragma unroll
    for (int u = 0; u < NORM_PASSES; ++u) {
      if (group * NORM_PASSES + u >= passes) break;
      bool in;
      const int k = column(group, u, in);
      room[(((group % 2) * NORM_PASSES + u) * SLICES + own) * NORM_PITCH + at] = in ? v[u] : f32x4{0.f, 0.f, 0.f, 0.f};
      if (in) *(f32x4*)(H + (size_t)m * K + k) = v[u] * g[u];
    }
    if (group + 1 < groups) load(group + 1);
    __syncthreads();                                    // (the first wave reads one half while the others fill the other)
    if (threadIdx.x < 32) {
#pragma unroll 1
      for (int u = 0; u < min(NORM_PASSES, passes - group * NORM_PASSES); ++u) {
        f32x4 q[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) q[x] = room[(((group % 2) * NORM_PASSES + u) * SLICES + threadIdx.x / 4) * NORM_PITCH + threadIdx.x % 4 + 4 * x];
#pragma unroll
        for (int x = 0; x < 8; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss[e % 2] = fmaf(q[x][e], q[x][e], ss[e % 2]);
      }
    }
  }
  if (threadIdx.x >= 32) return;
  float sum = ss[0] + ss[1];
  sum += __shfl_xor(sum, 1), sum += __shfl_xor(sum, 2);
  float all = 0.f;
#pragma unroll
  for (int w = 0; w < SLICES; ++w) all += __shfl(sum, w * 4, 32);
  if (threadIdx.x == 0) R[m] = row_scale(all, K, eps);
}

// MT x NT tiles of 16 rows x 16 outputs a block, D stages of loads ahead.
// GLU: W is [2 N][K], rows of gates and then rows of values; a block's bands of W are NT / 2 of gates and the NT / 2 of
// values that belong to them, and it writes silu(gate) * value.  A product is the same sum as without, so the result is
// the bits of the product of 2 N outputs and the activation's own pass.
// NORMALISED: A is the row in front of an RMS norm of weight G.  Every block reads whole rows of A anyway (a wave its own k), so a
// wave multiplies its operands by G, adds up the squares beside that, and the sums are scaled by the row's 1 / sqrt(mean
// square + eps) where the waves meet.  The squares of a row are added in an order that depends on K alone, too.  For one row
// tile only: with several, every block does it again for the same rows (325 rows x 8,192 outputs of SwiGLU 194 -> 205 us,
// twice the norm's own launch), so norm_rows_f32_kernel does it once, with the same operations, and R has the rows' scales (SCALED; a form
// of its own: with the scales' loads in front of every tile, behind a condition, the compiler waited there and where the waves
// meet for all that was on its way).
enum Rows { PLAIN, SCALED, NORMALISED };
template <int SL, int MT, int NT, int D, bool ONCE, int MIN_WAVES, bool GLU, int ROWS, bool ON>
__global__ __launch_bounds__(64 * SL, MIN_WAVES) void gemm_f32_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ G, float eps, const float* __restrict__ R,
    const float* __restrict__ W, int ldw, void* __restrict__ C, int c_dtype, int ldc, int M, int N, int K, int mode, int tiles_m, int tiles) {
  constexpr int BANDS = MT + NT;
  constexpr bool NORM = ROWS == NORMALISED;
  static_assert(!(ON && NORM), "the norm is in the product of one row tile only");
  constexpr int STAGE_F4 = BANDS * 128, SUM_F4 = MT * NT * 64;       // float4 a wave: its stage, and at the end its sums
  constexpr int WAVE_F4 = STAGE_F4 > SUM_F4 ? STAGE_F4 : SUM_F4;
  __shared__ f32x4 lds[SL * WAVE_F4];
  __shared__ float squares[NORM ? SL * 16 * MT : 1];
  __shared__ f32x4 gains[NORM ? NORM_K / 4 : 1];
  // The block ids that one XCD gets (every eighth) take a run of tiles, row tiles of the same outputs next to each other:
  // they share W in that XCD's L2.  A block goes on to the tile gridDim.x / 8 further in its run.
  const int per = (tiles + 7) / 8, first = (blockIdx.x % 8) * per, last = min(tiles, first + per), stride = gridDim.x / 8;
  int t = first + blockIdx.x / 8;
  if (t >= last) return;
  constexpr int NO = GLU ? NT / 2 : NT;                              // bands of outputs
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;

  const int slice = STAGE * ((K + STAGE * SLICES - 1) / (STAGE * SLICES));
  const int k0 = wave * slice;
  const int steps = (min(K, k0 + slice) - k0 + STAGE - 1) / STAGE;   // <= 0: no k left for this wave

  // What this lane loads of a stage: rows lane/8 and lane/8 + 8 of every band, 4 k at (lane%8)*4.  Rows past the end are
  // the last row again (their sums are not stored); for k past the end it loads the stage's first k, and 0 goes into LDS.
  const int lr = lane / 8, lk = (lane % 8) * 4;
  BufferRsrc from_w, from_a;
  int off[BANDS][2], m0, n0;
  auto aim = [&](int tile) __attribute__((always_inline)) {          // the loads that follow are of this tile
    m0 = (tile % tiles_m) * (16 * MT), n0 = (tile / tiles_m) * (16 * NO);
    const int rows_w = min(N - n0, 16 * NO), rows_a = min(M - m0, 16 * MT);
    from_w = make_rsrc(W + (size_t)n0 * ldw), from_a = make_rsrc(A + (size_t)m0 * lda);
#pragma unroll
    for (int b = 0; b < BANDS; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        off[b][h] = 4 * (lk + (b < NT ? ((b < NO ? 0 : N) + min(16 * (b % NO) + lr + 8 * h, rows_w - 1)) * ldw : min(16 * (b - NT) + lr + 8 * h, rows_a - 1) * lda));
  };
  f32x4 reg[D][BANDS][2];
  auto load_one = [&](int slot, int s, int b, int h) __attribute__((always_inline)) {
    const int at = 4 * (k0 + s * STAGE);
    const int back = k0 + s * STAGE + lk >= K ? 4 * lk : 0;
    reg[slot][b][h] = b < NT ? load_f32x4<ONCE>(from_w, off[b][h] - back, at) : load_f32x4<false>(from_a, off[b][h] - back, at);
  };
  float ss[NORM ? MT : 1][2];                           // squares of row lane % 16 of a band of A, of the k that this lane holds
  // G goes into LDS behind the first stages' loads: in registers beside every stage in flight it cost the tiles of few rows
  // their second block a unit.
  f32x4 gain[NORM ? NORM_K / (256 * SL) : 1] = {};
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NORM_K / (256 * SL); ++q)
      if (threadIdx.x + q * 64 * SL < K / 4) gain[q] = reinterpret_cast<const f32x4*>(G)[threadIdx.x + q * 64 * SL];
  }
  auto gains_in = [&]() __attribute__((always_inline)) {
    if constexpr (NORM) {
#pragma unroll
      for (int q = 0; q < NORM_K / (256 * SL); ++q) gains[threadIdx.x + q * 64 * SL] = gain[q];
      __syncthreads();
    }
  };
  auto load = [&](int slot, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BANDS; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) load_one(slot, s, b, h);
  };

  // the wave's stage in LDS: row r of a band is 8 pieces of 16 bytes, piece c at place c ^ (r % 8) (reads of one piece
  // over eight rows then fall on different banks)
  f32x4* mine = lds + wave * WAVE_F4;
  const int put_at = lr * 8 + ((lane % 8) ^ lr);
  const int row = lane % 16, quarter = lane / 16;
  const int get_at[2] = {row * 8 + (quarter ^ (row % 8)), row * 8 + ((quarter + 4) ^ (row % 8))};
  auto put_one = [&](int slot, int b, int h) __attribute__((always_inline)) { mine[b * 128 + h * 64 + put_at] = reg[slot][b][h]; };
  auto put_end = [&](int s) __attribute__((always_inline)) {
    if (k0 + (s + 1) * STAGE > K && k0 + s * STAGE + lk >= K) {
#pragma unroll
      for (int b = 0; b < 2 * BANDS; ++b) mine[b * 64 + put_at] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    wave_lds_order();
  };
  auto put = [&](int slot, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BANDS; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) put_one(slot, b, h);
    put_end(s);
  };
  f32x4 f[2][BANDS], g[NORM ? 2 : 1];                   // operands of a stage's first and second 16 k, the gains of those
  auto get = [&](int half, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BANDS; ++b) f[half][b] = mine[b * 128 + get_at[half]];
    if constexpr (NORM) g[half] = gains[(k0 + s * STAGE) / 4 + quarter + 4 * half];
    wave_lds_order();
  };
  auto normalise = [&](int half) __attribute__((always_inline)) {      // (zeros past the end of a row)
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ss[i][e % 2] = fmaf(f[half][NT + i][e], f[half][NT + i][e], ss[i][e % 2]);
          f[half][NT + i][e] *= g[half][e];
        }
    }
  };
  floatx4 acc[MT][NT];
  auto multiply_one = [&](int half, int u) __attribute__((always_inline)) {            // the u-th product of a half
    const int e = u / (MT * NT), i = u / NT % MT, j = u % NT;
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[half][j][e], f[half][NT + i][e], acc[i][j], 0, 0, 0);
  };
  constexpr int PRODUCTS = 4 * MT * NT;
  auto multiply = [&](int half) __attribute__((always_inline)) {
    normalise(half);
#pragma unroll
    for (int u = 0; u < PRODUCTS; ++u) multiply_one(half, u);
  };
  // The waves meet: their sums into LDS, then a thread adds the slices' sums of the pieces of four outputs that it stores.
  constexpr int PIECES = (MT * NO + SL - 1) / SL;
  auto meet = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) lds[wave * WAVE_F4 + (i * NT + j) * 64 + lane] = acc[i][j];
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float own = ss[i][0] + ss[i][1];
        own += __shfl_xor(own, 16), own += __shfl_xor(own, 32);
        if (quarter == 0) squares[wave * 16 * MT + i * 16 + row] = own;
      }
    }
    __syncthreads();
  };
  auto scale_of = [&](int q, int row0) __attribute__((always_inline)) {                // (SCALED)
    return R[min(row0 + (int)(threadIdx.x + q * 64 * SL) / (NO * 64) * 16 + (int)threadIdx.x % 16, M - 1)];
  };
  auto piece = [&](int q, float scale) __attribute__((always_inline)) {
    const int p = threadIdx.x + q * 64 * SL, i = p / (NO * 64), j = p / 64 % NO, l = p % 64;
    auto sum = [&](int band) __attribute__((always_inline)) {
      const int at = (i * NT + band) * 64 + l;
      f32x4 u = lds[at];
#pragma unroll
      for (int w = 1; w < SL; ++w) u += lds[w * WAVE_F4 + at];
      return u;
    };
    if constexpr (NORM) {
      float all = 0.f;
#pragma unroll
      for (int w = 0; w < SL; ++w) all += squares[w * 16 * MT + i * 16 + l % 16];
      scale = row_scale(all, K, eps);
    }
    f32x4 v = sum(j);
    if constexpr (ROWS != PLAIN) v *= scale;
    if constexpr (GLU) {
      f32x4 u = sum(NO + j);
      if constexpr (ROWS != PLAIN) u *= scale;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (v[e] / (1.0f + expf(-v[e]))) * u[e];
    }
    return v;
  };
  const bool wide = mode == 0 && c_dtype == APC_F32 && ldc % 4 == 0 && ((uintptr_t)C & 15u) == 0;   // 16-byte stores
  auto leave = [&](int q, const f32x4& v, int row0, int out0) __attribute__((always_inline)) {
    const int p = threadIdx.x + q * 64 * SL;
    const int m = row0 + p / (NO * 64) * 16 + p % 16, n = out0 + p / 64 % NO * 16 + (p % 64 / 16) * 4;
    if (m >= M) return;
    if (wide && n + 4 <= N) {
      *(f32x4*)((float*)C + (size_t)m * ldc + n) = v;
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (n + e >= N) continue;
      const size_t o = (size_t)m * ldc + n + e;
      if (mode == 1) ((float*)C)[o] += v[e];
      else store_f(C, c_dtype, o, v[e]);
    }
  };
  auto has = [&](int q) __attribute__((always_inline)) { return (int)threadIdx.x + q * 64 * SL < MT * NO * 64; };
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < MT; ++i) ss[i][0] = ss[i][1] = 0.f;
    }
  };

  aim(t);
  clear();
  // A stage: its second operands come out of LDS under the first products; then the next stage goes in, the loads that
  // take its registers go out, and its first operands come back under the second products.
  // Products, a piece's store and its load stand in this order, held by barriers of the scheduler: with the load's address worked
  // out in front of the store (the compiler's choice, which a change elsewhere in the kernel may move) the same instructions
  // take 2-4 % longer: 325 rows x 2,048 outputs x K 8,192 101.9 -> 98.9 us, 2,048 rows 527 -> 512, 325 x 8,192 SwiGLU 190.7 -> 185.8.
  if constexpr (ON) {
    // A block of these takes tile after tile.  Behind a tile's last stage its registers ask for the next tile's first one,
    // which is there when the eight waves have met; a launch of several rounds then pays the way of the first loads (every
    // wave's stage at once: 112 KB a unit), the block's start and the stores' way once and not every round.
    int at_stage = 0, at_tile = t;                      // the stage that the next load is of, and its tile
    auto asked = [&]() __attribute__((always_inline)) {
      if (++at_stage == steps) {
        at_stage = 0;
        if (at_tile + stride < last) aim(at_tile += stride);         // (no tile left: a stage that nobody takes)
      }
    };
    auto first_in = [&]() __attribute__((always_inline)) {
      put(0, 0);
      __builtin_amdgcn_sched_barrier(0);
      load(0, at_stage);
      __builtin_amdgcn_sched_barrier(0);
      asked();
      get(0, 0);
    };
    int row0 = m0, out0 = n0;                           // of the tile that is multiplied
    if (steps > 0) load(0, 0), asked(), first_in();
    while (true) {
      if (steps > 0) {
        for (int s = 0; s < steps - 1; ++s) {
          get(1, s);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < 2 * BANDS; ++u) {
#pragma unroll
            for (int p = u * PRODUCTS / (2 * BANDS); p < (u + 1) * PRODUCTS / (2 * BANDS); ++p) multiply_one(0, p);
            __builtin_amdgcn_sched_barrier(0);
            put_one(0, u / 2, u % 2);
            __builtin_amdgcn_sched_barrier(0);
            load_one(0, at_stage, u / 2, u % 2);
            __builtin_amdgcn_sched_barrier(0);
          }
          put_end(s + 1);
          asked();
          get(0, s + 1);
          __builtin_amdgcn_sched_barrier(0);
          multiply(1);
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_waitcnt(0xc07f);           // LDS only
        }
        get(1, steps - 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        multiply(1);
      }
      t += stride;
      f32x4 v[PIECES];
      float scale[PIECES] = {};
      if constexpr (ROWS == SCALED)
#pragma unroll
        for (int q = 0; q < PIECES; ++q) scale[q] = scale_of(q, row0);
      meet();
#pragma unroll
      for (int q = 0; q < PIECES; ++q)
        if (has(q)) v[q] = piece(q, scale[q]);
      if (t < last) {
        __syncthreads();                                // everyone has read the sums
        clear();
        if (steps > 0) first_in();
      }
#pragma unroll
      for (int q = 0; q < PIECES; ++q)
        if (has(q)) leave(q, v[q], row0, out0);
      if (t >= last) break;
      row0 = (t % tiles_m) * (16 * MT), out0 = (t / tiles_m) * (16 * NO);
    }
  } else {
    float scale[PIECES] = {};
    if constexpr (ROWS == SCALED)
#pragma unroll
      for (int q = 0; q < PIECES; ++q) scale[q] = scale_of(q, m0);
    auto stage = [&](int s, int next_slot, bool next, bool more) __attribute__((always_inline)) {
      get(1, s);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      if (next) {
        put(next_slot, s + 1);
        __builtin_amdgcn_sched_barrier(0);                // (the loads take the registers that have just been written out)
        if (more) load(next_slot, s + 1 + D);
        __builtin_amdgcn_sched_barrier(0);
        get(0, s + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(1);
    };
    auto begin = [&](auto count) __attribute__((always_inline)) {                        // stages there are, at least (what is known when compiling)
      constexpr int R = decltype(count)::value;
#pragma unroll
      for (int u = 0; u < D && u < R; ++u) load(u, u);
      gains_in();
      put(0, 0);
      if (R > D) load(0, D);
      get(0, 0);
    };
    auto finish = [&](int s0, auto count) __attribute__((always_inline)) {               // the last stages, without a condition between the loads
      constexpr int R = decltype(count)::value;
#pragma unroll
      for (int i = 0; i < R; ++i) stage(s0 + i, (i + 1) % D, i + 1 < R, i + 1 + D < R);
    };
    // Straight code for the last 2 D stages: behind a branch that may have loaded the compiler waits for more than it needs.
    if (steps > 2 * D) {
      begin(Count<2 * D + 1>{});
      int s0 = 0;
      for (; steps - s0 > 2 * D; s0 += D)
#pragma unroll
        for (int u = 0; u < D; ++u) stage(s0 + u, (u + 1) % D, true, true);
      each_count<2 * D>([&](auto r) __attribute__((always_inline)) {
        if (steps - s0 == decltype(r)::value) finish(s0, r);
      });
    } else {
      each_count<2 * D>([&](auto r) __attribute__((always_inline)) {
        if (steps == decltype(r)::value) begin(r), finish(0, r);
      });
      if (steps <= 0) gains_in();
    }
    meet();
#pragma unroll
    for (int q = 0; q < PIECES; ++q)
      if (has(q)) leave(q, piece(q, scale[q]), m0, n0);
  }
}

// What goes with the product for q, k and v (ROPE): W is [(H + 2 Hk) d, K], heads in the order q, k, v, d a multiple of 16.  A block
// takes eight outputs j 8 .. of a head's first half and the same of its second, so that a lane of the first wave finds both elements of
// four pairs (e, e + d / 2) in the sums.  Rotated q goes to C; k to cache[page][0][kv head][slot][:], v to cache[page][1][kv
// head][:][slot], page = block_table[row_seg][pos / P], slot = pos % P.
struct RopeF32 {
  const float* cos_sin;     // [positions][2][d / 2]
  const int* positions;     // [M]
  const int* row_seg;       // [M]
  const int* block_table;   // [segments][max_blocks]
  int max_blocks;
  float* cache;
  int P, H, Hk, d;
};

// The product of up to 8 rows.  The same slices, the same sums to the bit as gemm_f32_kernel's; what differs is what a stage brings:
// 8 rows of A, not 16 of which half are repeats, and 8 rows of W (16 with ROPE), so that 2,048 outputs have a block for every unit;
// two stages are on their way in a loop whose last round asks again for the last stage instead of code for every remainder, and a
// stage's operands come out of LDS under the products of the one before.  A residual is asked for ahead of the first weights.
// What bounds it is a unit's eight waves' way from loads to products (as many stages as registers hold are no faster: 4 rows x
// 2,048 outputs x K 2,048 7.6 us with two, 7.9 with four, 8.7 with eight).  apc_gemm_f32_few says where it is taken, with both sides' times.
template <int BAND, int D, bool NORM, bool ROPE>
__global__ __launch_bounds__(64 * SLICES, 4) void gemm_f32_few_kernel(const float* __restrict__ A, int lda, const float* __restrict__ G,
                                                                      float eps, const float* __restrict__ W, int ldw, void* __restrict__ C,
                                                                      int c_dtype, int ldc, int M, int N, int K, int mode, RopeF32 rope) {
  static_assert(!ROPE || BAND == 16, "two halves of eight");
  static_assert(D % 2 == 0 && (BAND == 8 || BAND == 16), "two stages in LDS take turns");
  constexpr int WL = BAND / 8, STAGE_F4 = 64 * (WL + 1);
  __shared__ f32x4 lds[SLICES][2][STAGE_F4];
  __shared__ float squares[NORM ? SLICES * 16 : 1];
  __shared__ f32x4 gains[NORM ? NORM_K / 4 : 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int slice = STAGE * ((K + STAGE * SLICES - 1) / (STAGE * SLICES)), k0 = wave * slice;
  const int steps = (min(K, k0 + slice) - k0 + STAGE - 1) / STAGE;   // <= 0: no k left for this wave
  const int lr = lane / 8, lk = (lane % 8) * 4, row = lane % 16, quarter = lane / 16;
  const int head = ROPE ? blockIdx.x / (rope.d / 16) : 0, j = ROPE ? blockIdx.x % (rope.d / 16) : 0, half_head = rope.d / 2;
  const int n0 = ROPE ? head * rope.d + j * 8 : blockIdx.x * BAND;
  const BufferRsrc from_w = make_rsrc(W + (size_t)n0 * ldw), from_a = make_rsrc(A);
  int off[WL + 1];
#pragma unroll
  for (int h = 0; h < WL; ++h) off[h] = 4 * ((ROPE ? h * half_head + lr : min(8 * h + lr, N - 1 - n0)) * ldw + lk);
  off[WL] = 4 * (min(lr, M - 1) * lda + lk);
  // the outputs that a lane of the first wave leaves: row `row`, n .. n + 3
  const int n = n0 + quarter * 4;
  const bool own = wave == 0 && row < M && quarter * 4 < (ROPE ? 8 : BAND);
  const bool wide = c_dtype == APC_F32 && ldc % 4 == 0 && ((uintptr_t)C & 15u) == 0 && n + 4 <= N;   // 16 bytes
  f32x4 before = {0.f, 0.f, 0.f, 0.f};
  if (own && wide && mode == 1) before = *(const f32x4*)((const float*)C + (size_t)row * ldc + n);
  int pos = 0, seg = 0, page = 0;                       // ROPE: asked for in front of the first weights, what hangs on them behind
  f32x4 cs = {0.f, 0.f, 0.f, 0.f}, sn = {0.f, 0.f, 0.f, 0.f};
  if (ROPE && own) pos = rope.positions[row], seg = rope.row_seg[row];
  f32x4 reg[D][WL + 1];
  auto load = [&](int slot, int s) __attribute__((always_inline)) {
    s = min(s, steps - 1);
    const int at = 4 * (k0 + s * STAGE), back = k0 + s * STAGE + lk >= K ? 4 * lk : 0;
#pragma unroll
    for (int h = 0; h < WL; ++h) reg[slot][h] = load_f32x4<true>(from_w, off[h] - back, at);
    reg[slot][WL] = load_f32x4<false>(from_a, off[WL] - back, at);
  };
  const int put_at = lr * 8 + ((lane % 8) ^ lr);
  auto put = [&](int slot, int s, int to) __attribute__((always_inline)) {
    const bool end = k0 + min(s, steps - 1) * STAGE + lk >= K;       // (behind K: zeros)
#pragma unroll
    for (int h = 0; h <= WL; ++h) lds[wave][to][h * 64 + put_at] = end ? f32x4{0.f, 0.f, 0.f, 0.f} : reg[slot][h];
    wave_lds_order();
  };
  f32x4 w[2][2], a[2][2], g[2][2];                      // [stage % 2][half]: operands, gains of the stage's 16 k
  auto get = [&](int s, int from) __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int piece = (quarter + 4 * half) ^ (row % 8);
      w[from][half] = lds[wave][from][row % BAND * 8 + piece];
      a[from][half] = lds[wave][from][WL * 64 + row % 8 * 8 + piece];
      if constexpr (NORM) g[from][half] = gains[(k0 + min(s, steps - 1) * STAGE) / 4 + quarter + 4 * half];
    }
    wave_lds_order();
  };
  float ss[2] = {0.f, 0.f};
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int of) __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ss[e % 2] = fmaf(a[of][half][e], a[of][half][e], ss[e % 2]), a[of][half][e] *= g[of][half][e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[of][half][e], a[of][half][e], acc, 0, 0, 0);
    }
  };
  f32x4 gain[NORM ? NORM_K / (256 * SLICES) : 1] = {};
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NORM_K / (256 * SLICES); ++q)
      if (threadIdx.x + q * 64 * SLICES < K / 4) gain[q] = reinterpret_cast<const f32x4*>(G)[threadIdx.x + q * 64 * SLICES];
  }
  if (steps > 0) {
#pragma unroll
    for (int u = 0; u < D; ++u) load(u, u);
  }
  if (ROPE && own) {
    const float* at = rope.cos_sin + (size_t)pos * rope.d + j * 8 + quarter * 4;
    cs = *(const f32x4*)at, sn = *(const f32x4*)(at + half_head);
    page = rope.block_table[(size_t)seg * rope.max_blocks + pos / rope.P];
  }
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NORM_K / (256 * SLICES); ++q) gains[threadIdx.x + q * 64 * SLICES] = gain[q];
    __syncthreads();
  }
  if (steps > 0) {
    put(0, 0, 0);
    load(0, D);
    get(0, 0);
    for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        put((u + 1) % D, s0 + u + 1, (u + 1) % 2);
        load((u + 1) % D, s0 + u + 1 + D);
        get(s0 + u + 1, (u + 1) % 2);
        if (s0 + u < steps) multiply(u % 2);
      }
    }
  }
  lds[wave][0][lane] = acc;                             // the waves meet
  if constexpr (NORM) {
    float sq = ss[0] + ss[1];
    sq += __shfl_xor(sq, 16), sq += __shfl_xor(sq, 32);
    if (quarter == 0) squares[wave * 16 + row] = sq;
  }
  __syncthreads();
  if (!own) return;
  auto sum = [&](int l) __attribute__((always_inline)) {
    f32x4 v = lds[0][0][l];
#pragma unroll
    for (int x = 1; x < SLICES; ++x) v += lds[x][0][l];
    return v;
  };
  float scale = 1.f;
  if constexpr (NORM) {
    float all = 0.f;
#pragma unroll
    for (int x = 0; x < SLICES; ++x) all += squares[x * 16 + row];
    scale = row_scale(all, K, eps);
  }
  f32x4 v = sum(lane);
  if constexpr (NORM) v *= scale;
  if constexpr (ROPE) {
    f32x4 hi = sum(lane + 32);
    if constexpr (NORM) hi *= scale;
    const int e = j * 8 + quarter * 4, slot = pos % rope.P;
    float* in_page = rope.cache + (size_t)page * ((size_t)2 * rope.Hk * rope.P * rope.d);
    if (head < rope.H + rope.Hk) {
      f32x4 ra, rb;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float fa = v[x], fb = hi[x], c = cs[x], s = sn[x];
        ra[x] = fmaf(fa, c, -(fb * s));                 // (as the compiler makes it of rope_kv_write_kernel's text)
        rb[x] = fmaf(fb, c, fa * s);
      }
      float* to = head < rope.H ? (float*)C + (size_t)row * ldc + (size_t)head * rope.d
                                : in_page + ((size_t)(head - rope.H) * rope.P + slot) * rope.d;
      *(f32x4*)(to + e) = ra;
      *(f32x4*)(to + e + half_head) = rb;
    } else {
      float* to = in_page + ((size_t)(rope.Hk + head - rope.H - rope.Hk) * rope.d + e) * rope.P + slot;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        to[(size_t)x * rope.P] = v[x];
        to[(size_t)(half_head + x) * rope.P] = hi[x];
      }
    }
    return;
  }
  if (wide) {
    *(f32x4*)((float*)C + (size_t)row * ldc + n) = mode == 1 ? before + v : v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (n + e >= N) continue;
    const size_t o = (size_t)row * ldc + n + e;
    if (mode == 1) ((float*)C)[o] += v[e];
    else store_f(C, c_dtype, o, v[e]);
  }
}

// Slices without k are left out: with all eight, a block of a large tile keeps its unit for 6 us whatever K is, most of
// its waves idle and 128 KiB of LDS taken.  2,048 rows x 16,384 outputs at K = 32, 64, 128: 200, 203, 216 us with eight
// slices and stores of 4 bytes, 84, 101, 147 with the two or four there are, 53, 69, 125 with 16-byte stores beside (one
// fma chain an output on the vector units: 70, 98, 150).
template <int SL, int MT, int NT, int D, bool ONCE, int MIN_WAVES, bool GLU, int ROWS, bool ON>
int launch_slices(const float* A, int lda, const float* G, float eps, const float* R, const float* W, int ldw, void* C,
                  int c_dtype, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
  const int tiles_m = ceil_div(M, 16 * MT);
  const long long tiles = (long long)tiles_m * ceil_div(N, 16 * (GLU ? NT / 2 : NT));
  if (tiles > (1 << 27)) return APC_ERR_BAD_ARG;
  int blocks = ceil_div((int)tiles, 8) * 8;
  if (ON && blocks > 256) blocks = 256;                 // such a block has a compute unit to itself
  hipLaunchKernelGGL((gemm_f32_kernel<SL, MT, NT, D, ONCE, MIN_WAVES, GLU, ROWS, ON>), dim3(blocks), dim3(64 * SL), 0,
                     stream, A, lda, G, eps, R, W, ldw, C, c_dtype, ldc, M, N, K, mode, tiles_m, (int)tiles);
  APC_LAUNCH_CHECK();
  return 0;
}

// Which tiles' blocks go on to further tiles, with a stage's stores and loads between its products.  Time of the form that ends
// after its tile / of this one, mean over 17 to 2,048 rows x 64 to 32,768 outputs: 32 x 32 tiles (two blocks a unit without it)
// 0.87-0.95 at every K; 48 x 32 in one round of 256 blocks 0.91-0.99, in more 1.05-1.09 up to K = 1,024 and 1.00-1.03 beyond;
// 48 x 64 one round 0.92-0.98 up to K = 512, 1.02-1.04 beyond, more rounds 1.01-1.10; 64 x 64 0.84-0.97 up to K = 512, then one
// round 0.97 up to K = 1,024, else 1.00-1.02.  SwiGLU: 48 x 16 outputs 0.93-1.00, the others as their products.
bool goes_on(int mt, int nt, bool glu, int M, int N, int K) {
  const bool rounds = (long long)ceil_div(M, 16 * mt) * ceil_div(N, 16 * (glu ? nt / 2 : nt)) > 256;
  if (K <= 4 * STAGE || mt * nt < 6 || (mt * nt == 6 && glu)) return false;
  return mt * nt == 6 ? rounds : mt * nt == 12 ? rounds || K > 512 : K > (rounds ? 512 : 1024);
}

template <int MT, int NT, int D, bool ONCE, int MIN_WAVES, bool GLU = false>
int launch(const float* A, int lda, const float* G, float eps, const float* R, const float* W, int ldw, void* C, int c_dtype,
           int ldc, int M, int N, int K, int mode, hipStream_t stream) {
  if constexpr (MT == 1 && ONCE)
    if (G) return launch_slices<SLICES, MT, NT, D, ONCE, MIN_WAVES, GLU, NORMALISED, false>(A, lda, G, eps, R, W, ldw, C, c_dtype, ldc, M, N, K, mode, stream);
  if (G) return APC_ERR_UNSUPPORTED;
#define SL_GO(SL_, ON_)                                                                                                             \
  return R ? launch_slices<SL_, MT, NT, D, ONCE, MIN_WAVES, GLU, SCALED, ON_>(A, lda, G, eps, R, W, ldw, C, c_dtype, ldc, M, N, K, mode, stream) \
           : launch_slices<SL_, MT, NT, D, ONCE, MIN_WAVES, GLU, PLAIN, ON_>(A, lda, G, eps, R, W, ldw, C, c_dtype, ldc, M, N, K, mode, stream)
  if constexpr (MT * NT >= 4 && MT * NT <= 6) {         // (smaller tiles share their units with eight too; larger ones are not chosen)
    if (K <= 2 * STAGE) SL_GO(2, false);
    if (K <= 4 * STAGE) SL_GO(4, false);
  }
  if constexpr (MT * NT > 6 || (MT * NT == 6 && !GLU))
    if (goes_on(MT, NT, GLU, M, N, K)) SL_GO(SLICES, true);
  SL_GO(SLICES, false);
#undef SL_GO
}

}  // namespace

// Whether the kernel takes these operands: 16-byte loads along k.
bool gemm_f32_takes(const void* A, int lda, const void* W, int ldw, int K) {
  return K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15u) == 0 && lda < (1 << 22) &&
         ldw < (1 << 22);            // (64 rows fit a descriptor's 32-bit offsets)
}

// A tile of 16 mt x 16 nt and what a launch of its blocks costs, in microseconds: once, and for every 256 of them (a round); each
// a part that stays and a part that grows with K, as for K = 2,048.  `part`: how far a last round that is not full takes less
// (1: blocks share their units, their time grows with them).  `over`: what the columns up to the next multiple of 256 count (a K
// between leaves waves with a stage less than the others).
struct TileCost { int mt, nt; double start, start_k, round, round_k, over, part; };
template <int COUNT>
static int least_cost(const TileCost (&shapes)[COUNT], int M, int N, int K, int outputs) {   // outputs: of 16 nt columns
  int best = 0;
  double best_cost = 1e30;
  for (int i = 0; i < COUNT; ++i) {
    const TileCost& s = shapes[i];
    const double raw = (double)ceil_div(M, 16 * s.mt) * ceil_div(N, outputs * s.nt) / 256;
    const double rounds = raw > 1.0 ? s.part * raw + (1.0 - s.part) * ceil(raw) : 1.0;
    const double k = (K + s.over * (SLICES * STAGE * ceil_div(K, SLICES * STAGE) - K)) / 2048;
    const double cost = s.start + s.start_k * k + (s.round + s.round_k * k) * rounds;
    if (cost < best_cost) best = i, best_cost = cost;
  }
  return best;
}

// The tile: the least expected time.  Fitted to 2,233 products of 17 to 2,048 rows x 64 to 32,768 outputs, K 160 to 14,336, each on
// all six tiles: the choice takes 1.008 of the best tile's time in the mean, more than 1.03 in 199 of them, 1.22 at worst (100
// rows x 6,144 outputs, K = 512: 16.4 us, 13.4 on 64 x 64).  K = 2,048: 33 rows x 2,048 outputs 10.1 us (32 x 16 tiles; 32 x 32 13.1),
// 325 rows 30.6 (48 x 64), 2,048 rows 146 (64 x 64; 48 x 64 159); K = 256: 64 rows x 16,384 10.1 (64 x 64).
// Up to K = 128 (see launch) blocks of all tiles share their units, and with many outputs tiles that leave the empty slices out
// are the better ones for few rows too: 16 rows x 128,256 outputs, 32 x 32 / 16 x 16 tiles, K = 32 10.4 / 19.6 us, 64 13.1 / 22.6, 128
// 22.2 / 25.7; 32,768 outputs 4.5 / 6.7, 5.2 / 7.1.
constexpr TileCost TILES[] = {{1, 1, 0.45, 1.86, 1.48, 4.05, 0.4, 0.77},   {2, 1, 1.74, 1.19, 0.85, 5.6, 0.4, 0.07},
                              {2, 2, 3.18, 0.71, 0.74, 9.07, 0.55, 0.11},  {3, 2, 1.98, 0.79, 1.37, 13.92, 0.55, 0.07},
                              {3, 4, 2.43, 1.29, 2.41, 24.83, 0.55, 0.09}, {4, 4, 2.39, 0.61, 3.7, 33.4, 0.55, 0.18}};
constexpr TileCost TILES_SHORT[] = {{1, 1, 3.6, 0.0, 0.75, 0.0, 0.0, 1.0}, {2, 1, 3.6, 0.0, 0.95, 0.0, 0.0, 1.0}, {2, 2, 4.1, 0.0, 0.69, 0.0, 0.0, 1.0},
                                    {3, 2, 4.4, 0.0, 0.93, 0.0, 0.0, 1.0}};        // (48 x 64 and 64 x 64 are never the least)
static int tile_of(int M, int N, int K) {
  if (K <= 4 * STAGE) return least_cost(TILES_SHORT, M, N, K, 16);
  return M <= 16 ? 0 : least_cost(TILES, M, N, K, 16);   // (the other tiles multiply rows that are not there)
}

// Rows of the tile, times 1,000, and its outputs.
APC_EXPORT int apc_gemm_f32_tile(int M, int N, int K) {
  const TileCost& t = TILES[tile_of(M, N, K)];
  return 16 * t.mt * 1000 + 16 * t.nt;
}

// Tiles that a block of the product takes at most: 1 where it ends behind its tile.
static int tiles_a_block(const TileCost& t, bool glu, int M, int N, int K) {
  const int tiles = ceil_div(M, 16 * t.mt) * ceil_div(N, 16 * (glu ? t.nt / 2 : t.nt));
  return goes_on(t.mt, t.nt, glu, M, N, K) ? ceil_div(ceil_div(tiles, 8), 32) : 1;
}
APC_EXPORT int apc_gemm_f32_tiles_a_block(int M, int N, int K) { return tiles_a_block(TILES[tile_of(M, N, K)], false, M, N, K); }

// Whether a product without a norm goes to gemm_f32_few_kernel: up to 8 rows, one round of blocks of 8 outputs, and a short K only
// where the sums are added to what is there, which is then asked for early.  Launches of a graph over 0.5 GB of weights, tiles / blocks
// of 8 outputs, us, 4 rows (1 and 8 rows within 5 % of it), stored: 2,048 outputs x K 2,048 6.6 / 6.4, K 8,192 19.7 / 18.3, 1,024 x
// 4,096 9.6 / 9.0, but 2,048 x 256 3.4 / 3.6, x 1,024 4.7 / 4.9; added: 2,048 x 256 3.8 / 3.8, x 2,048 7.1 / 6.7, x 8,192 20.3 / 18.5, 1,024
// x 4,096 10.1 / 9.1, 576 x 576 4.7 / 4.3.  Beyond 2,048 outputs blocks of 16 lost, stored: 3,072 x 2,048 7.0 / 7.4, 4,096 x 1,028 6.5 /
// 7.6, 4,096 x 4,096 13.1 / 13.5 (added: 13.4 / 13.5).
APC_EXPORT int apc_gemm_f32_few(int M, int N, int K, int mode) {
  return M > 0 && M <= 8 && N > 0 && N <= 2048 && K > (mode == 1 ? 4 * STAGE : 1024) ? 1 : 0;
}

// Few rows: two stages of loads ahead, not four.  4 rows x 2,048 outputs x K 2,048 7.2 -> 6.7 us, K 8,192 21.6 -> 19.3 (128,256
// outputs, K 2,048: 150 and 151): the straight code of a stage count's every case is a third as long, and a launch finds it cold.
static int product(const float* A, int lda, const float* G, float eps, const float* R, const float* W, int ldw, void* C,
                   int c_dtype, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
  if (!G && !R && apc_gemm_f32_few(M, N, K, mode)) {
    hipLaunchKernelGGL((gemm_f32_few_kernel<8, 2, false, false>), dim3(ceil_div(N, 8)), dim3(64 * SLICES), 0, stream, A, lda, nullptr, 0.f,
                       W, ldw, C, c_dtype, ldc, M, N, K, mode, RopeF32{});
    APC_LAUNCH_CHECK();
    return 0;
  }
#define GO(...) return launch<__VA_ARGS__>(A, lda, G, eps, R, W, ldw, C, c_dtype, ldc, M, N, K, mode, stream)
  // (one row tile: W is read once, past the caches)
  switch (tile_of(M, N, K)) {
    case 0:
      if (M <= 16) GO(1, 1, 2, true, 4);
      GO(1, 1, 4, false, 4);
    case 1:
      if (M <= 32) GO(2, 1, 2, true, 2);
      GO(2, 1, 2, false, 2);
    case 2: GO(2, 2, 1, false, 2);
    case 3: GO(3, 2, 1, false, 2);
    case 4: GO(3, 4, 1, false, 2);
    default: GO(4, 4, 1, false, 2);
  }
#undef GO
}

int gemm_f32(const float* A, int lda, const float* W, int ldw, void* C, int c_dtype, int ldc, int M, int N, int K, int mode,
             hipStream_t stream) {
  return product(A, lda, nullptr, 0.f, nullptr, W, ldw, C, c_dtype, ldc, M, N, K, mode, stream);
}

// C[M,N] = rmsnorm(A; G, eps) . W^T.  Up to 16 rows in one launch: 4 rows x 3,072 outputs x K 2,048 7.1 us without the norm, 7.6
// with it, and the norm's own launch was 4.7; 6,144 x K 4,096 21.6 and 21.0.  More rows need room for M rows of K and their
// scales: apc_gemm_norm_f32_kib(M, K) KiB; they buy the bits of the few rows, not time (325 rows x 3,072 outputs 51 us, the norm's launch
// and the product 5 and 46).  A row's outputs do not depend on the rows beside it, nor on M.
// With a short K and many outputs every block does the norm again for little else: 8 rows x 128,256 outputs, in the product / in
// front of it, K = 256 44.1 / 32.2 us, 512 62.2 / 45.6, 1,024 90.9 / 80.1 (2,048 on: the other way), 32,768 outputs 13.1 / 12.1,
// 18.1 / 16.1, 26.1 / 26.0, 14,336 outputs 9.9 / 10.3 at K = 512; SwiGLU at K = 512 of 32,768 outputs 28.1 / 28.3, of 128,256 95.0 / 89.1.
static bool norm_in_product(int M, int N, int K, int tile, int most) { return M <= 16 && K <= NORM_K && (K > 1024 || N <= most) && tile == 0; }
APC_EXPORT int apc_gemm_norm_f32_kib(int M, int K) {
  return M <= 16 && K > 1024 && K <= NORM_K ? 0 : (int)(((long long)M * (K + 1) * 4 + 1023) / 1024);
}
APC_EXPORT int apc_gemm_norm_f32_takes(const void* A, int lda, const void* G, const void* W, int ldw, int K) {
  return gemm_f32_takes(A, lda, W, ldw, K) && G && ((uintptr_t)G & 15u) == 0;
}
static int norm_rows(const float* A, int lda, const float* G, float eps, float* ws, int M, int K, hipStream_t stream) {
  if (!ws || ((uintptr_t)ws & 15u)) return APC_ERR_BAD_ARG;
  // Two rows a wave / a row a block, us: 17 rows of 512 2.3 / 2.4, of 2,048 2.8 / 2.6, of 4,096 3.9 / 3.1, of 8,192 6.2 / 4.4; 177 of
  // 4,096 5.2 / 4.1; 330 of 2,048 4.1 / 4.1; 1,024 of 2,048 6.7 / 7.7, of 8,192 17.2 / 12.7; 2,048 of 1,024 6.3 / 8.4.
  if (K > NORM_K || (M <= 512 && K > 512)) {
    const int passes = ceil_div(STAGE * ceil_div(K, STAGE * SLICES), 128);
    const int lds = (passes < 2 * NORM_PASSES ? passes : 2 * NORM_PASSES) * SLICES * NORM_PITCH * 16;
    hipLaunchKernelGGL(norm_row_f32_kernel, dim3(M), dim3(256), lds, stream, A, lda, G, eps, ws, ws + (size_t)M * K, M, K);
  } else {
    hipLaunchKernelGGL(norm_rows_f32_kernel, dim3(ceil_div(M, 2)), dim3(64), 0, stream, A, lda, G, eps, ws, ws + (size_t)M * K, M, K);
  }
  APC_LAUNCH_CHECK();
  return 0;
}

APC_EXPORT int apc_gemm_norm_f32(const void* A, int lda, const void* G, float eps, const void* W, int ldw, void* C, int ldc, int M,
                                 int N, int K, void* ws, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldc < N) return APC_ERR_BAD_ARG;
  if (!apc_gemm_norm_f32_takes(A, lda, G, W, ldw, K)) return APC_ERR_UNSUPPORTED;
  const float *a = (const float*)A, *g = (const float*)G, *w = (const float*)W;
  if (norm_in_product(M, N, K, tile_of(M, N, K), 16384)) return product(a, lda, g, eps, nullptr, w, ldw, C, APC_F32, ldc, M, N, K, 0, stream);
  float* h = (float*)ws;
  if (const int rc = norm_rows(a, lda, g, eps, h, M, K, stream)) return rc;
  return product(h, K, nullptr, 0.f, h + (size_t)M * K, w, ldw, C, APC_F32, ldc, M, N, K, 0, stream);
}

// q, k and v of up to 8 rows in one launch with the norm in front, the rotation of whole q and k heads and the write of k and v into
// the pages (see RopeF32); q_out [M, ldq] takes the rotated q heads in its first H d columns.  The sums are apc_gemm_norm_f32's.
// 4 rows of a 1B model (3,072 outputs, K 2,048), inside a step: 8.4 + 4.6 -> 9.6 us.  Up to 8,192 outputs: from there on the tiles are
// faster by what the launch costs.
APC_EXPORT int apc_qkv_rope_f32_takes(const void* A, int lda, const void* G, const void* W, int ldw, const void* q_out, int ldq, int M,
                                      int K, int H, int Hk, int d, const void* cos_sin, const void* cache) {
  if (M <= 0 || M > 8 || H <= 0 || Hk <= 0 || d <= 0 || d % 16 || (H + 2 * Hk) * (long long)d > 8192) return 0;
  if (K <= 4 * STAGE || K > NORM_K || lda < K || ldw < K || ldq < H * d || ldq % 4) return 0;
  if ((((uintptr_t)q_out | (uintptr_t)cos_sin | (uintptr_t)cache) & 15u) || (d / 2 + 8LL) * ldw * 4 >= (1LL << 31)) return 0;
  return apc_gemm_norm_f32_takes(A, lda, G, W, ldw, K);
}
APC_EXPORT int apc_qkv_rope_f32(const float* A, int lda, const float* G, float eps, const float* W, int ldw, float* q_out, int ldq, int M,
                                int K, int H, int Hk, int d, const float* cos_sin, const int* positions, const int* row_seg,
                                const int* block_table, int max_blocks, float* cache, int page_tokens, hipStream_t stream) {
  if (M <= 0) return 0;
  if (!positions || !row_seg || !block_table || max_blocks <= 0 || !cache || !cos_sin || page_tokens <= 0) return APC_ERR_BAD_ARG;
  if (!apc_qkv_rope_f32_takes(A, lda, G, W, ldw, q_out, ldq, M, K, H, Hk, d, cos_sin, cache)) return APC_ERR_UNSUPPORTED;
  const RopeF32 rope{cos_sin, positions, row_seg, block_table, max_blocks, cache, page_tokens, H, Hk, d};
  hipLaunchKernelGGL((gemm_f32_few_kernel<16, 2, true, true>), dim3((H + 2 * Hk) * d / 16), dim3(64 * SLICES), 0, stream, A, lda, G, eps, W,
                     ldw, q_out, APC_F32, ldq, M, (H + 2 * Hk) * d, K, 0, rope);
  APC_LAUNCH_CHECK();
  return 0;
}

// out[M,F] = silu(A . Wg^T) * (A . Wu^T), W = [Wg; Wu] of 2 F rows: the same sums as the product of 2 F outputs, without
// the pass over them (4.8 us of a layer of 4 rows x 8,192, 7 of one of 340): both products and the activation take 22.6 us
// with 4 rows of K = 2,048 and 210 with 340.
APC_EXPORT int apc_swiglu_f32_takes(const void* A, int lda, const void* W, int ldw, int F, int K) {
  return gemm_f32_takes(A, lda, W, ldw, K) && ((long long)F + 64) * ldw < (1LL << 29);   // byte offsets of 32 bits
}

// (1,801 gated products of 17 to 1,024 rows x 64 to 14,336 outputs, K 160 to 8,192: 1.004 of the best tile's time in the mean, 1.10
// at worst.  K = 2,048, 8,192 outputs: 325 rows 186 us on 48 x 32 tiles, 205 on 48 x 16, 211 on 64 x 32; 100 rows 76 on 64 x 32, 85 on 48 x 32.)
constexpr TileCost GLU_TILES[] = {{1, 2, 2.44, 2.65, 0.55, 5.34, 0.4, 0.16}, {2, 2, 3.03, 1.13, 0.83, 8.93, 0.55, 0.44},
                                  {3, 2, 2.82, 0.89, 1.1, 14.48, 0.55, 0.39}, {3, 4, 2.49, 1.85, 2.2, 24.42, 0.55, 0.0},
                                  {4, 4, 0.55, 1.13, 3.44, 32.83, 0.55, 0.0}};
constexpr TileCost GLU_TILES_SHORT[] = {{1, 2, 3.6, 0.0, 0.95, 0.0, 0.0, 1.0}, {2, 2, 4.1, 0.0, 0.69, 0.0, 0.0, 1.0}, {3, 2, 4.4, 0.0, 0.93, 0.0, 0.0, 1.0}};
static int glu_tile_of(int M, int F, int K) {
  if (K <= 4 * STAGE) return least_cost(GLU_TILES_SHORT, M, F, K, 8);
  return M <= 16 ? 0 : least_cost(GLU_TILES, M, F, K, 8);
}

// Rows of the tile, times 1,000, and its outputs (half of the columns it computes).
APC_EXPORT int apc_swiglu_f32_tile(int M, int F, int K) {
  const TileCost& t = GLU_TILES[glu_tile_of(M, F, K)];
  return 16 * t.mt * 1000 + 8 * t.nt;
}

APC_EXPORT int apc_swiglu_f32_tiles_a_block(int M, int F, int K) { return tiles_a_block(GLU_TILES[glu_tile_of(M, F, K)], true, M, F, K); }

static int swiglu(const void* A, int lda, const void* G, float eps, const float* R, const void* W, int ldw, void* out, int ldo,
                  int M, int F, int K, hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldo < F) return APC_ERR_BAD_ARG;
  if (!apc_swiglu_f32_takes(A, lda, W, ldw, F, K)) return APC_ERR_UNSUPPORTED;
#define GO(...)                                                                                                             \
  return launch<__VA_ARGS__, true>((const float*)A, lda, (const float*)G, eps, R, (const float*)W, ldw, out, APC_F32, ldo, M, F, K, \
                                   0, stream)
  switch (glu_tile_of(M, F, K)) {
    case 0:
      if (M <= 16) GO(1, 2, 2, true, 4);
      GO(1, 2, 2, false, 4);
    case 1: GO(2, 2, 1, false, 2);
    case 2: GO(3, 2, 1, false, 2);
    case 3: GO(3, 4, 1, false, 2);
    default: GO(4, 4, 1, false, 2);
  }
#undef GO
}

APC_EXPORT int apc_swiglu_f32(const void* A, int lda, const void* W, int ldw, void* out, int ldo, int M, int F, int K,
                              hipStream_t stream) {
  return swiglu(A, lda, nullptr, 0.f, nullptr, W, ldw, out, ldo, M, F, K, stream);
}

// The same of the normalised rows, out of the rows in front of the norm (4 rows x 8,192 outputs x K 2,048: 22.6 us without the
// norm, 23.8 with it); the workspace is apc_gemm_norm_f32's.
APC_EXPORT int apc_swiglu_norm_f32_takes(const void* A, int lda, const void* G, const void* W, int ldw, int F, int K) {
  return apc_swiglu_f32_takes(A, lda, W, ldw, F, K) && G && ((uintptr_t)G & 15u) == 0;
}

APC_EXPORT int apc_swiglu_norm_f32(const void* A, int lda, const void* G, float eps, const void* W, int ldw, void* out, int ldo,
                                   int M, int F, int K, void* ws, hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldo < F) return APC_ERR_BAD_ARG;
  if (!apc_swiglu_norm_f32_takes(A, lda, G, W, ldw, F, K)) return APC_ERR_UNSUPPORTED;
  if (norm_in_product(M, F, K, glu_tile_of(M, F, K), 32768)) return swiglu(A, lda, G, eps, nullptr, W, ldw, out, ldo, M, F, K, stream);
  float* h = (float*)ws;
  if (const int rc = norm_rows((const float*)A, lda, (const float*)G, eps, h, M, K, stream)) return rc;
  return swiglu(h, K, nullptr, 0.f, h + (size_t)M * K, W, ldw, out, ldo, M, F, K, stream);
}
