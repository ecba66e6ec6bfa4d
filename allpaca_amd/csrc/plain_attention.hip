// Plain attention over the paged cache.  This first kernel takes any types and sizes: one wave per (query row, head),
// keys in order in chunks of 64 anchored at key 0, online softmax in float32.  (float32 queries and pages in pieces of
// 16 bytes: paged_attention_f32_kernel below, which adds in another fixed order.)
//
// For the row at position `pos` of its request:  keys t in [first, pos],
// first = 0 or pos - window + 1;  s_t = (q . K[t]) * scale;  m = max s;
// p_t = exp(s_t - m);  out = sum p_t V[t] / sum p_t;  query head h reads kv head
// h / (H/Hk).  Reference: crates/allpaca-cpu/src/kernels.rs:293-356 (the causal
// rule `t <= qi + (n_kv - n_q)` is `t <= pos` once rows carry their position);
// the chunked online form follows hip/src/kernels.cpp:1917-1934 in spirit: the
// order of additions for a row is fixed by its position alone, never by what
// else is in the batch or how the prompt was cut.
//
// keys cache[page][0][kv_head][slot][i], values cache[page][1][kv_head][i][slot];
// page = block_table[seg][t / P], slot = t % P.
#include "common.h"
#include <math.h>

constexpr int MAX_D_PER_LANE = 4;  // head_dim <= 256

__global__ __launch_bounds__(64) void paged_attention_plain_kernel(
    const void* __restrict__ q, int q_dtype, int ldq, int q_off, void* __restrict__ out, int out_dtype, int ldo, int H,
    int Hk, int d, const void* __restrict__ cache, int cache_dtype, int P, const int* __restrict__ block_table,
    int max_blocks, const int* __restrict__ positions, const int* __restrict__ row_seg, int window, float scale) {
  __shared__ float qs[MAX_D_PER_LANE * WAVE];
  __shared__ float ps[WAVE];
  const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int kvh = h / (H / Hk);
  const int pos = positions[r];
  const int* bt = block_table + (size_t)row_seg[r] * max_blocks;
  const int first = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;

  for (int i = lane; i < d; i += WAVE) qs[i] = load_f(q, q_dtype, (size_t)r * ldq + q_off + (size_t)h * d + i);
  __syncthreads();

  float o[MAX_D_PER_LANE];
#pragma unroll
  for (int i = 0; i < MAX_D_PER_LANE; ++i) o[i] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int c = first / WAVE; c <= pos / WAVE; ++c) {
    const int t = c * WAVE + lane;
    const bool valid = t >= first && t <= pos;
    float s = -INFINITY;
    if (valid) {
      const int page = bt[t / P];
      const size_t kb = ((((size_t)page * 2 + 0) * Hk + kvh) * P + (t % P)) * d;
      float dot = 0.f;
      for (int i = 0; i < d; ++i) dot = fmaf(qs[i], load_f(cache, cache_dtype, kb + i), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));  // finite: every chunk in the range holds a valid key
    const float alpha = expf(m - m_new);        // exp(-inf) = 0 on the first chunk
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int i = 0; i < MAX_D_PER_LANE; ++i) o[i] *= alpha;
    __syncthreads();
    ps[lane] = p;
    __syncthreads();
    const int j_end = min(WAVE, pos - c * WAVE + 1);
    const int j_begin = max(0, first - c * WAVE);
    for (int j = j_begin; j < j_end; ++j) {
      const float pj = ps[j];
      const int tj = c * WAVE + j;
      const int page = bt[tj / P];
      const size_t vb = (((size_t)page * 2 + 1) * Hk + kvh) * (size_t)P * d + (tj % P);
#pragma unroll
      for (int i = 0; i < MAX_D_PER_LANE; ++i) {
        const int e = lane + i * WAVE;
        if (e < d) o[i] = fmaf(pj, load_f(cache, cache_dtype, vb + (size_t)e * P), o[i]);
      }
    }
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < MAX_D_PER_LANE; ++i) {
    const int e = lane + i * WAVE;
    if (e < d) store_f(out, out_dtype, (size_t)r * ldo + (size_t)h * d + e, o[i] * inv);
  }
}

// The same for float32 queries and a float32 cache whose head size and page size are multiples of 4.  A row's chunks of
// 64 keys go to eight lists (chunk c to list c % 8), each with an online softmax of its own, and the lists' results are
// added in order at the end: a row's additions again depend on its position alone.  Against the kernel above: a key is
// read 16 bytes a load and once for the HB heads that share it, a value likewise four slots at a time.  Two forms with
// the same arithmetic:
//   SPREAD   a block of eight waves a row, a wave a list: few rows (decoding), where the chain position -> page -> keys ->
//            softmax -> values of a chunk, about 4 us, is what takes the time; all of a chunk's values are asked for
//            before its keys.
//   else     a block of four waves, a row each, one list after the other: many rows (prompts), where the number of
//            loads is; waves that have no chunk would stand idle in the other form.
// Measured, 32 heads of 64 on 8 kv heads, microseconds a layer (the kernel above): 4 rows at 101 to 907 keys 15 (259),
// 340 rows of three prompts 33 (205).  Prompts on the SPREAD form: 73.  With heads over 64 in groups of 4 the SPREAD form
// is 6 registers short and keeps them in scratch memory (32 heads of 128 on 8 kv heads, 4 rows at 100 to 900
// keys: 33 us, 523 in the kernel above).
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int LISTS = 8, ROWS_A_BLOCK = 4;

template <int HB, int EL>
struct ListState {                 // HB heads, EL elements of a head a lane
  float o[HB][EL], m[HB], l[HB];
};

struct AttArgs {
  const float* q;
  int ldq, q_off;
  float* out;
  int ldo, H, Hk, d;
  const float* cache;
  int P;
  const int* block_table;
  int max_blocks;
  const int *positions, *row_seg;
  int window;
  float scale;
  int n_rows;
};

// One chunk of one list.  qs: the row's HB query heads; ps: room for the chunk's weights.
template <int HB, int EL, bool AHEAD>
__device__ __forceinline__ void attend_chunk(const AttArgs& A, int kvh, const int* bt, int first, int pos, int c, const f32x4* qs,
                                             f32x4 (*ps)[WAVE / 4], ListState<HB, EL>& S) {
  const int lane = threadIdx.x % WAVE, d = A.d, P = A.P, d4 = d / 4;
  const int t = c * WAVE + lane;
  const bool valid = t >= first && t <= pos;
  const int tv = min(max(t, first), pos);                // (a key that is there, for lanes without one)
  const int page = bt[tv / P];
  // The page size is a multiple of 4, so the four slots of a load lie in one page: that of their first key, or of the
  // nearest key that is there.
  auto values = [&](int j, f32x4* v) __attribute__((always_inline)) {
    const int vp = __builtin_amdgcn_readlane(page, 4 * j);
    const float* at = A.cache + (((size_t)vp * 2 + 1) * A.Hk + kvh) * (size_t)P * d + (c * WAVE + 4 * j) % P;
#pragma unroll
    for (int i = 0; i < EL; ++i) v[i] = *(const f32x4*)(at + (size_t)(lane + i * WAVE < d ? lane + i * WAVE : 0) * P);
  };
  constexpr int N = AHEAD ? WAVE / 4 : 4;                // loads of values that are out together
  f32x4 v[N][EL];
  if (AHEAD)
#pragma unroll
    for (int j = 0; j < N; ++j) values(j, v[j]);
  const f32x4* k = (const f32x4*)(A.cache + ((((size_t)page * 2 + 0) * A.Hk + kvh) * P + (tv % P)) * d);
  float dot[HB];
#pragma unroll
  for (int h = 0; h < HB; ++h) dot[h] = 0.f;
  int i0 = 0;
  for (; i0 + 8 <= d4; i0 += 8) {
    f32x4 kv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) kv[u] = k[i0 + u];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int h = 0; h < HB; ++h) {
        const f32x4 qv = qs[h * d4 + i0 + u];
#pragma unroll
        for (int e = 0; e < 4; ++e) dot[h] = fmaf(qv[e], kv[u][e], dot[h]);
      }
  }
  for (; i0 < d4; ++i0) {
    const f32x4 kv = k[i0];
#pragma unroll
    for (int h = 0; h < HB; ++h) {
      const f32x4 qv = qs[h * d4 + i0];
#pragma unroll
      for (int e = 0; e < 4; ++e) dot[h] = fmaf(qv[e], kv[e], dot[h]);
    }
  }
  float p[HB];
#pragma unroll
  for (int h = 0; h < HB; ++h) {
    const float s = valid ? dot[h] * A.scale : -INFINITY;
    const float m_new = fmaxf(S.m[h], wave_max(s));      // finite: every chunk in the range holds a valid key
    const float alpha = expf(S.m[h] - m_new);             // exp(-inf) = 0 on the first chunk
    p[h] = valid ? expf(s - m_new) : 0.f;
    S.l[h] = fmaf(S.l[h], alpha, wave_sum(p[h]));
    S.m[h] = m_new;
#pragma unroll
    for (int i = 0; i < EL; ++i) S.o[h][i] *= alpha;
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int h = 0; h < HB; ++h) ((float*)ps[h])[lane] = p[h];
  __builtin_amdgcn_wave_barrier();
  const int from = first - c * WAVE, to = pos - c * WAVE;  // the keys the row sees; other slots may hold anything
  auto add = [&](int j, const f32x4* x4) __attribute__((always_inline)) {
    f32x4 pj[HB];
#pragma unroll
    for (int h = 0; h < HB; ++h) pj[h] = ps[h][j];
#pragma unroll
    for (int i = 0; i < EL; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float x = 4 * j + u >= from && 4 * j + u <= to ? x4[i][u] : 0.f;
#pragma unroll
        for (int h = 0; h < HB; ++h) S.o[h][i] = fmaf(pj[h][u], x, S.o[h][i]);
      }
  };
  if (AHEAD) {
#pragma unroll
    for (int j = 0; j < N; ++j) add(j, v[j]);
  } else {
    for (int j0 = 0; j0 < WAVE / 4; j0 += N) {
      if (4 * j0 > to || 4 * (j0 + N) <= from) {         // none of these keys: what `add` would do with weights of 0
#pragma unroll
        for (int h = 0; h < HB; ++h)
#pragma unroll
          for (int i = 0; i < EL; ++i) S.o[h][i] += 0.f;
        continue;
      }
#pragma unroll
      for (int j = 0; j < N; ++j) values(j0 + j, v[j]);
#pragma unroll
      for (int j = 0; j < N; ++j) add(j0 + j, v[j]);
    }
  }
}

template <int HB, int EL, bool SPREAD>
__global__ __launch_bounds__((SPREAD ? LISTS : ROWS_A_BLOCK) * WAVE) void paged_attention_f32_kernel(AttArgs A) {
  constexpr int WAVES = SPREAD ? LISTS : ROWS_A_BLOCK, ROWS = SPREAD ? 1 : ROWS_A_BLOCK;
  __shared__ f32x4 qs[ROWS][HB * EL * WAVE / 4];
  __shared__ f32x4 ps[WAVES][HB][WAVE / 4];
  __shared__ float ends[ROWS][LISTS][HB][2];
  __shared__ float os[ROWS][LISTS][HB][EL * WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int at = SPREAD ? 0 : wave;                       // the row's place in LDS
  const int r = SPREAD ? blockIdx.x : blockIdx.x * ROWS + wave;
  if (r >= A.n_rows) return;                              // (without SPREAD: no barrier below)
  const int h0 = blockIdx.y * HB, kvh = h0 / (A.H / A.Hk), d = A.d;
  const int pos = A.positions[r];
  const int* bt = A.block_table + (size_t)A.row_seg[r] * A.max_blocks;
  const int first = (A.window > 0 && pos - A.window + 1 > 0) ? pos - A.window + 1 : 0;
  const int part = SPREAD ? threadIdx.x : lane, parts = SPREAD ? WAVES * WAVE : WAVE;   // of the threads on this row
  for (int i = part; i < HB * d; i += parts) ((float*)qs[at])[i] = A.q[(size_t)r * A.ldq + A.q_off + (size_t)h0 * d + i];
  if (SPREAD) __syncthreads();
  else __builtin_amdgcn_wave_barrier();

  const int c0 = first / WAVE, c1 = pos / WAVE;
  auto list = [&](int w) __attribute__((always_inline)) {
    ListState<HB, EL> S;
#pragma unroll
    for (int h = 0; h < HB; ++h) {
      S.m[h] = -INFINITY;
      S.l[h] = 0.f;
#pragma unroll
      for (int i = 0; i < EL; ++i) S.o[h][i] = 0.f;
    }
    for (int c = c0 + (w - c0 % LISTS + LISTS) % LISTS; c <= c1; c += LISTS)
      attend_chunk<HB, EL, SPREAD>(A, kvh, bt, first, pos, c, qs[at], ps[wave], S);
#pragma unroll
    for (int h = 0; h < HB; ++h) {
      if (lane == 0) ends[at][w][h][0] = S.m[h], ends[at][w][h][1] = S.l[h];
#pragma unroll
      for (int i = 0; i < EL; ++i) os[at][w][h][lane + i * WAVE] = S.o[h][i];
    }
  };
  if (SPREAD) {
    list(wave);
    __syncthreads();
  } else {
    for (int w = 0; w < LISTS; ++w) list(w);
    __builtin_amdgcn_wave_barrier();
  }
  for (int i = part; i < HB * d; i += parts) {
    const int h = i / d, e = i % d;
    float mm = -INFINITY, ll = 0.f, oo = 0.f;
    for (int w = 0; w < LISTS; ++w) mm = fmaxf(mm, ends[at][w][h][0]);
    for (int w = 0; w < LISTS; ++w) {
      const float f = expf(ends[at][w][h][0] - mm);       // (0 for a list without keys)
      ll = fmaf(ends[at][w][h][1], f, ll);
      oo = fmaf(os[at][w][h][e], f, oo);
    }
    A.out[(size_t)r * A.ldo + (size_t)h0 * d + i] = oo * (1.0f / ll);
  }
}

template <int HB, int EL>
void launch_f32(const AttArgs& A, hipStream_t stream) {
  // up to two blocks of the spread form a compute unit: one a row and HB heads
  const int blocks = A.H / HB;
  if ((long long)A.n_rows * blocks <= 512)
    hipLaunchKernelGGL((paged_attention_f32_kernel<HB, EL, true>), dim3(A.n_rows, blocks), dim3(LISTS * WAVE), 0, stream, A);
  else
    hipLaunchKernelGGL((paged_attention_f32_kernel<HB, EL, false>), dim3(ceil_div(A.n_rows, ROWS_A_BLOCK), blocks),
                       dim3(ROWS_A_BLOCK * WAVE), 0, stream, A);
}

// While every row and head can have a compute unit to itself, blocks of one head, even where four share a kv head: a
// chunk's arithmetic stands between its loads, and what is then read four times comes out of L2.  The heads' sums are the
// same.  32 heads on 8 kv heads, 4 rows at 101 to 907 keys: heads of 64 18.2 -> 16.2 us, of 128 34.3 -> 28.6; 8 rows at 900
// keys 19.0 -> 16.9 and 49.2 -> 36.0; 16 rows at 900 keys would go from 23.9 to 34.2 and from 51.3 to 68.5.
// Long contexts too, where the bytes go past the L2 of one XCD: it is the units that are few, not the bytes.  8 rows at 8,192
// and 24,000 keys, each from pages that no launch has just read: heads of 64 191 -> 151 and 544 -> 426 us, of 128 460 -> 355 and
// 1,337 -> 1,023.  Over 1 to 10 rows of 130 to 24,000 keys, groups of 2 to 8 heads, 0.72 to 1.05 of the time, 0.88 in the mean.
template <int EL>
void launch_heads(const AttArgs& A, hipStream_t stream) {
  const int group = A.H / A.Hk;
  if ((long long)A.n_rows * A.H <= 256 || group % 2) launch_f32<1, EL>(A, stream);
  else if (group % 4) launch_f32<2, EL>(A, stream);
  else launch_f32<4, EL>(A, stream);
}

APC_EXPORT int apc_paged_attention_plain(const void* q, int q_dtype, int ldq, int q_off, void* out, int out_dtype,
                                         int ldo, int n_rows, int H, int Hk, int d, const void* cache,
                                         int cache_dtype, int page_tokens, const int* block_table, int max_blocks,
                                         const int* positions, const int* row_seg, int window, float scale,
                                         hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (H <= 0 || Hk <= 0 || H % Hk || d <= 0 || page_tokens <= 0 || max_blocks <= 0 || window < 0)
    return APC_ERR_BAD_ARG;
  if (d > MAX_D_PER_LANE * WAVE || H > 65535) return APC_ERR_UNSUPPORTED;
  // float32 in 16-byte pieces: by types, sizes and strides only, so that a row does not depend on the batch
  if (q_dtype == APC_F32 && out_dtype == APC_F32 && cache_dtype == APC_F32 && d % 4 == 0 && d <= 2 * WAVE &&
      page_tokens % 4 == 0 && ((uintptr_t)cache & 15u) == 0) {
    const AttArgs A{(const float*)q, ldq,       q_off,       (float*)out, ldo,    H,     Hk,    d, (const float*)cache,
                    page_tokens,     block_table, max_blocks, positions,   row_seg, window, scale, n_rows};
    if (d <= WAVE) launch_heads<1>(A, stream);
    else launch_heads<2>(A, stream);
    APC_LAUNCH_CHECK();
    return 0;
  }
  hipLaunchKernelGGL(paged_attention_plain_kernel, dim3(n_rows, H), dim3(64), 0, stream, q, q_dtype, ldq, q_off, out,
                     out_dtype, ldo, H, Hk, d, cache, cache_dtype, page_tokens, block_table, max_blocks, positions,
                     row_seg, window, scale);
  APC_LAUNCH_CHECK();
  return 0;
}
