// The gated linear recurrence (see plain_delta.hip for the formulas) over prompt portions, bfloat16 rows, chunks of 64
// rows side by side, each in 4 runs of 16.  S_t = a_t S_(t-1) + b_t is linear in S, so three launches replace the walk
// row by row:
//   summaries  every run for itself, from a state of zero: its end state E and the sum of its log a; a block's 4 runs
//              are put together to the chunk's
//   scan       per segment and channel: the state in front of every chunk, S0_(k+1) = exp(sum_k) S0_k + E_k, starting
//              from the request's state, which is left at the segment's end
//   outputs    every run again from the state in front of it (the chunk's, carried over the runs ahead of it):
//              S_t * gelu(y_t) * out_scale
// A thread has two neighbouring channels of a run and asks for 8 rows of them at a time; a wave is a run.  All arithmetic
// is float32 (exponentials through the hardware's base-2 instruction, 1 - a^2 without cancellation); u, y and the output
// are bfloat16 rows, the gates' logits float32 rows.
#include "mfma.h"
#include <math.h>

namespace {

constexpr int CHUNK = 64;         // rows of a chunk (the step's list of chunks is made for this)
constexpr int RUNS = 4;           // runs of a chunk: the waves of a block
constexpr int RUN = CHUNK / RUNS;
constexpr int RU = 8;             // rows asked for together

__device__ __forceinline__ float sigmoid_fast(float z) { return 1.0f / (1.0f + __expf(-z)); }
// sqrt(1 - exp(x)), x <= 0: near 0 by the series of exp(x) - 1, which loses nothing to cancellation
__device__ __forceinline__ float root_rest(float x) {
  const float series = -x * (1.0f + x * (0.5f + x * (0.16666667f + x * (0.041666667f + x * 0.0083333333f))));
  return sqrtf(x > -0.1f ? series : 1.0f - __expf(x));
}

template <int MODE>   // 1: summaries, 2: outputs
__global__ __launch_bounds__(256) void recurrence_chunk_kernel(
    const bf16_t* __restrict__ u, int ldu, const float* __restrict__ z, int ldz, const float* __restrict__ zb, int w,
    const float* __restrict__ rate, const bf16_t* __restrict__ y, int ldy, const float* __restrict__ yb, float out_scale,
    float* __restrict__ ws, float* __restrict__ logs, float* __restrict__ run_e, float* __restrict__ run_l, int C,
    const int* __restrict__ chunks, const int* __restrict__ seg_row0, const int* __restrict__ seg_rows,
    bf16_t* __restrict__ out, int ldo) {
  __shared__ float4 sums[RUNS][WAVE];
  const int lane = threadIdx.x % WAVE, run = threadIdx.x / WAVE;
  const int c_own = (blockIdx.x * WAVE + lane) * 2, chunk = blockIdx.y;
  const bool on = c_own < C;
  const int c = on ? c_own : 0;                  // (the threads beyond the channels read channel 0 and store nothing)
  const int seg = chunks[2 * chunk], in_seg = chunks[2 * chunk + 1] + run * RUN;
  const int r0 = seg_row0[seg] + in_seg, n = min(RUN, seg_rows[seg] - in_seg);      // (n <= 0: a run without rows)
  const int zr = c / w * 2 * w + c % w, zi = zr + w;
  const float2 br = *reinterpret_cast<const float2*>(zb + zr), bi = *reinterpret_cast<const float2*>(zb + zi);
  const float2 k = *reinterpret_cast<const float2*>(rate + c);
  const float2 by = MODE == 2 && yb ? *reinterpret_cast<const float2*>(yb + c) : float2{0.f, 0.f};
  float2 S = float2{0.f, 0.f};
  if (MODE == 2) {
    S = *reinterpret_cast<const float2*>(ws + (size_t)chunk * C + c);
    for (int x = 0; x < run; ++x) {
      const size_t at = ((size_t)chunk * RUNS + x) * C + c;
      const float2 e = *reinterpret_cast<const float2*>(run_e + at), l = *reinterpret_cast<const float2*>(run_l + at);
      S.x = fmaf(__expf(l.x), S.x, e.x);
      S.y = fmaf(__expf(l.y), S.y, e.y);
    }
  }
  float2 total = float2{0.f, 0.f};
  for (int t0 = 0; t0 < n; t0 += RU) {
    float2 vr[RU], vi[RU];
    uint32_t vu[RU], vy[RU];
#pragma unroll
    for (int x = 0; x < RU; ++x) {
      const size_t row = r0 + min(t0 + x, n - 1);
      vr[x] = *reinterpret_cast<const float2*>(z + row * ldz + zr);
      vi[x] = *reinterpret_cast<const float2*>(z + row * ldz + zi);
      vu[x] = *reinterpret_cast<const uint32_t*>(u + row * ldu + c);
      if (MODE == 2) vy[x] = *reinterpret_cast<const uint32_t*>(y + row * ldy + c);
    }
#pragma unroll
    for (int x = 0; x < RU; ++x) {
      if (t0 + x >= n) break;
      const float l0 = k.x * sigmoid_fast(vr[x].x + br.x), l1 = k.y * sigmoid_fast(vr[x].y + br.y);
      const float i0 = sigmoid_fast(vi[x].x + bi.x) * __uint_as_float(vu[x] << 16);
      const float i1 = sigmoid_fast(vi[x].y + bi.y) * __uint_as_float(vu[x] & 0xffff0000u);
      S.x = fmaf(__expf(l0), S.x, root_rest(2.0f * l0) * i0);
      S.y = fmaf(__expf(l1), S.y, root_rest(2.0f * l1) * i1);
      total.x += l0;
      total.y += l1;
      if (MODE == 2) {
        const float g0 = activation_f(__uint_as_float(vy[x] << 16) + by.x, 3);
        const float g1 = activation_f(__uint_as_float(vy[x] & 0xffff0000u) + by.y, 3);
        if (on)
          *reinterpret_cast<uint32_t*>(out + (size_t)(r0 + t0 + x) * ldo + c) =
              pack_bf16x2(S.x * g0 * out_scale, S.y * g1 * out_scale);
      }
    }
  }
  if (MODE == 1) {
    sums[run][lane] = float4{S.x, S.y, total.x, total.y};
    __syncthreads();
    if (!on) return;
    const size_t at = ((size_t)chunk * RUNS + run) * C + c;
    *reinterpret_cast<float2*>(run_e + at) = S;
    *reinterpret_cast<float2*>(run_l + at) = total;
    if (run == 0) {
      float4 all = sums[0][lane];
#pragma unroll
      for (int x = 1; x < RUNS; ++x) {
        const float4 v = sums[x][lane];
        all = float4{fmaf(__expf(v.z), all.x, v.x), fmaf(__expf(v.w), all.y, v.y), all.z + v.z, all.w + v.w};
      }
      *reinterpret_cast<float2*>(ws + (size_t)chunk * C + c) = float2{all.x, all.y};
      *reinterpret_cast<float2*>(logs + (size_t)chunk * C + c) = float2{all.z, all.w};
    }
  }
}

// ws [chunks][C]: a chunk's end state in, the state in front of it out
__global__ __launch_bounds__(256) void recurrence_states_kernel(float* __restrict__ ws, const float* __restrict__ logs,
                                                                float* __restrict__ state,
                                                                const int* __restrict__ seg_chunks,
                                                                const int* __restrict__ slots, int C) {
  const int seg = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  const int k0 = seg_chunks[2 * seg], nk = seg_chunks[2 * seg + 1];
  float* st = state + (size_t)slots[seg] * C + c;
  float s = *st;
  for (int x0 = 0; x0 < nk; x0 += RU) {
    float e[RU], l[RU];
#pragma unroll
    for (int x = 0; x < RU; ++x) {
      const size_t at = (size_t)(k0 + min(x0 + x, nk - 1)) * C + c;
      e[x] = ws[at];
      l[x] = logs[at];
    }
#pragma unroll
    for (int x = 0; x < RU; ++x) {
      if (x0 + x >= nk) break;
      ws[(size_t)(k0 + x0 + x) * C + c] = s;
      s = fmaf(__expf(l[x]), s, e[x]);
    }
  }
  *st = s;
}

// ---- One row of every request (decoding): convolution, the gates' products and the recurrence in one launch ----
// A block takes one of the parts and all rows (up to 16): the convolution of its channels, moving the requests' kept inputs on,
// into LDS; a wave's bands of r's and i's logits on the matrix cores, their weights asked for at the very start; and where the
// logits lie, four channels of a row a lane, the recurrence, whose state, y and constants were asked for at the start too.  The
// operations are those of conv_channels_bf16x8_kernel, heads_gemm_few_kernel and gated_recurrence_kernel, in their order, so the
// results are the same bits.  What bounds it is latency: three launches that do this took 5.8 + 3.5 + 3.7 us for 8 rows of 2,048
// channels in 16 parts (1 MB of weights), this takes 7.0 (6.2 + 4.5 + 3.7 beside it); 25 steps of 8 requests 8.72 -> 8.48 ms.
constexpr int STEP_ROWS = 16, STEP_W = 256, STEP_PAD = 8, STEP_WAVES = 8;
__device__ __forceinline__ float sigmoid_exact(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float gelu_tanh_exact(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

struct StepArgs {
  const bf16_t *x, *y;             // [M][C] rows of strides ldx, ldy
  int ldx, ldy;
  const float *in_bias, *conv_w, *conv_b;
  float* conv_state;               // [slot][taps - 1][C]
  const bf16_t* W;                 // [parts][2 w / 16][w / 32] tiles
  const float *zb, *rate, *yb;
  float out_scale;
  float* state;                    // [slot][C]
  const int *row_seg, *conv_slots, *slots;
  bf16_t* out;
  int ldo, M, C, w;
};

template <int TAPS, int CHUNKS>    // CHUNKS: w / 32
__global__ __launch_bounds__(STEP_WAVES * 64) void recurrent_step_kernel(StepArgs A) {
  constexpr int w = CHUNKS * 32, BANDS = w / 16, TURNS = (BANDS + STEP_WAVES - 1) / STEP_WAVES;
  __shared__ __attribute__((aligned(16))) bf16_t us[STEP_ROWS][w + STEP_PAD];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, li = lane % 16, lc = lane / 16;
  const int part = blockIdx.x, c0 = part * w, row = min(li, A.M - 1);
  const bf16_t* wp = A.W + (size_t)part * 2 * BANDS * CHUNKS * 512 + lane * 8;
  Frag fr[CHUNKS], fi[CHUNKS];
  auto load_gates = [&](int band) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k) {
      fr[k] = load_frag(wp + (size_t)(band * CHUNKS + k) * 512);
      fi[k] = load_frag(wp + (size_t)((BANDS + band) * CHUNKS + k) * 512);
    }
  };
  load_gates(min(wave, BANDS - 1));
  const int slot = A.slots[A.row_seg[row]];

  for (int p = threadIdx.x; p < A.M * (w / 8); p += STEP_WAVES * 64) {
    const int r = p / (w / 8), c = c0 + p % (w / 8) * 8;
    float* st = A.conv_state + (size_t)A.conv_slots[A.row_seg[r]] * (TAPS - 1) * A.C + c;
    float u[TAPS][8], ib[8], b[8], wt[8][TAPS];
    const uint4 v = *reinterpret_cast<const uint4*>(A.x + (size_t)r * A.ldx + c);
#pragma unroll
    for (int j = 0; j + 1 < TAPS; ++j) {
      const float4 lo = *reinterpret_cast<const float4*>(st + (size_t)j * A.C), hi = *reinterpret_cast<const float4*>(st + (size_t)j * A.C + 4);
      u[j][0] = lo.x; u[j][1] = lo.y; u[j][2] = lo.z; u[j][3] = lo.w;
      u[j][4] = hi.x; u[j][5] = hi.y; u[j][6] = hi.z; u[j][7] = hi.w;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int j = 0; j < TAPS; ++j) wt[e][j] = A.conv_w[(size_t)(c + e) * TAPS + j];
      b[e] = A.conv_b ? A.conv_b[c + e] : 0.f;
      ib[e] = A.in_bias ? A.in_bias[c + e] : 0.f;
    }
    const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u[TAPS - 1][2 * k] = __uint_as_float(q[k] << 16) + ib[2 * k];
      u[TAPS - 1][2 * k + 1] = __uint_as_float(q[k] & 0xffff0000u) + ib[2 * k + 1];
    }
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      acc[e] = 0.f;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) acc[e] = fmaf(wt[e][j], u[j][e], acc[e]);     // oldest first
      if (A.conv_b) acc[e] += b[e];
    }
    *reinterpret_cast<uint4*>(&us[r][p % (w / 8) * 8]) =
        uint4{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]), pack_bf16x2(acc[4], acc[5]), pack_bf16x2(acc[6], acc[7])};
#pragma unroll
    for (int j = 1; j < TAPS; ++j) {
      *reinterpret_cast<float4*>(st + (size_t)(j - 1) * A.C) = float4{u[j][0], u[j][1], u[j][2], u[j][3]};
      *reinterpret_cast<float4*>(st + (size_t)(j - 1) * A.C + 4) = float4{u[j][4], u[j][5], u[j][6], u[j][7]};
    }
  }

  for (int turn = 0; turn < TURNS; ++turn) {
    const int band = wave + turn * STEP_WAVES;
    const bool on = band < BANDS && li < A.M;
    const int at = min(band, BANDS - 1) * 16 + lc * 4, c = c0 + at;     // this lane's first channel, in the part and in all
    float* sp = A.state + (size_t)slot * A.C + c;
    const float4 S4 = *reinterpret_cast<const float4*>(sp), k4 = *reinterpret_cast<const float4*>(A.rate + c);
    const float4 br4 = *reinterpret_cast<const float4*>(A.zb + 2 * c0 + at), bi4 = *reinterpret_cast<const float4*>(A.zb + 2 * c0 + w + at);
    const float4 by4 = A.yb ? *reinterpret_cast<const float4*>(A.yb + c) : float4{0.f, 0.f, 0.f, 0.f};
    const uint2 y2 = *reinterpret_cast<const uint2*>(A.y + (size_t)row * A.ldy + c);
    if (turn == 0) __syncthreads();                     // the convolution's rows are there
    floatx4 zr = floatx4{0.f, 0.f, 0.f, 0.f}, zi = zr;
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k) {
      const Frag fa = *reinterpret_cast<const Frag*>(&us[li][k * 32 + lc * 8]);   // (rows past the last hold anything: columns of their own)
      zr = mfma16(fr[k], fa, zr);
      zi = mfma16(fi[k], fa, zi);
    }
    if (turn + 1 < TURNS) load_gates(min(band + STEP_WAVES, BANDS - 1));
    if (!on) continue;
    const float Sv[4] = {S4.x, S4.y, S4.z, S4.w}, kv[4] = {k4.x, k4.y, k4.z, k4.w}, br[4] = {br4.x, br4.y, br4.z, br4.w};
    const float bi[4] = {bi4.x, bi4.y, bi4.z, bi4.w}, by[4] = {by4.x, by4.y, by4.z, by4.w};
    const uint2 u2 = *reinterpret_cast<const uint2*>(&us[li][at]);
    float S[4], o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t ub = e < 2 ? u2.x : u2.y, yw = e < 2 ? y2.x : y2.y;
      const float uv = __uint_as_float(e % 2 ? ub & 0xffff0000u : ub << 16), yv = __uint_as_float(e % 2 ? yw & 0xffff0000u : yw << 16);
      const float log_a = kv[e] * sigmoid_exact(zr[e] + br[e]);
      const float in = sigmoid_exact(zi[e] + bi[e]) * uv;
      S[e] = fmaf(expf(log_a), Sv[e], sqrtf(-expm1f(2.0f * log_a)) * in);
      o[e] = S[e] * gelu_tanh_exact(yv + by[e]) * A.out_scale;
    }
    *reinterpret_cast<float4*>(sp) = float4{S[0], S[1], S[2], S[3]};
    *reinterpret_cast<uint2*>(A.out + (size_t)li * A.ldo + c) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  }
}

}  // namespace

// 1 if the kernels take these sizes, else 0 (the caller then runs the kernel that walks row by row)
APC_EXPORT int apc_gated_recurrence_bf16_takes(int C, int blocks, int ldu, int ldz, int ldy, int ldo) {
  return (C > 0 && blocks > 0 && C % blocks == 0 && (C / blocks) % 2 == 0 && ldu % 2 == 0 && ldz % 2 == 0 && ldy % 2 == 0 &&
          ldo % 2 == 0) ? 1 : 0;
}

// chunks, seg_chunks: as in apc_delta_rule_bf16; work: float32 [10][n_chunks][C]
APC_EXPORT int apc_gated_recurrence_bf16(const void* u, int ldu, const float* z, int ldz, const float* zb, int blocks,
                                         const float* rate, const void* y, int ldy, const float* yb, float out_scale,
                                         float* state, int C, int n_segs, const int* seg_row0, const int* seg_rows,
                                         const int* slots, int n_chunks, const int* chunks, const int* seg_chunks,
                                         float* work, void* out, int ldo, hipStream_t stream) {
  if (n_segs <= 0 || n_chunks <= 0) return 0;
  if (!apc_gated_recurrence_bf16_takes(C, blocks, ldu, ldz, ldy, ldo)) return APC_ERR_UNSUPPORTED;
  if (!u || !z || !zb || !rate || !y || !state || !slots || !chunks || !seg_chunks || !work || !out || ldu < C ||
      ldz < 2 * C || ldy < C || ldo < C || ((uintptr_t)u & 3u) || ((uintptr_t)y & 3u) || ((uintptr_t)out & 3u) ||
      ((uintptr_t)z & 7u) || ((uintptr_t)work & 7u))
    return APC_ERR_BAD_ARG;
  if (n_chunks > 65535 || n_segs > 65535) return APC_ERR_UNSUPPORTED;
  const dim3 grid(ceil_div(C / 2, WAVE), n_chunks);
  const size_t part = (size_t)n_chunks * C;
  float *ws = work, *logs = work + part, *run_e = work + 2 * part, *run_l = run_e + RUNS * part;
#define REC_LAUNCH(MODE_)                                                                                              \
  hipLaunchKernelGGL(recurrence_chunk_kernel<MODE_>, grid, dim3(256), 0, stream, (const bf16_t*)u, ldu, z, ldz, zb,     \
                     C / blocks, rate, (const bf16_t*)y, ldy, yb, out_scale, ws, logs, run_e, run_l, C, chunks,        \
                     seg_row0, seg_rows, (bf16_t*)out, ldo);                                                                               \
  APC_LAUNCH_CHECK()
  REC_LAUNCH(1);
  hipLaunchKernelGGL(recurrence_states_kernel, dim3(ceil_div(C, 256), n_segs), dim3(256), 0, stream, ws, logs, state,
                     seg_chunks, slots, C);
  APC_LAUNCH_CHECK();
  REC_LAUNCH(2);
#undef REC_LAUNCH
  return 0;
}

// 1 if one launch takes a step of M single rows with these sizes and strides
APC_EXPORT int apc_recurrent_step_bf16_takes(int M, int C, int parts, int taps, int ldx, int ldy, int ldo) {
  if (M < 1 || M > STEP_ROWS || C <= 0 || parts <= 0 || C % parts || taps < 2 || taps > 4) return 0;
  const int w = C / parts;
  return ((w == 32 || w == 64 || w == 128 || w == 256) && w <= STEP_W && ldx % 8 == 0 && ldy % 4 == 0 && ldo % 4 == 0) ? 1 : 0;
}

// row_seg: a row's segment, of which it is the only row; conv_slots, slots: the segments' places in conv_state and state
APC_EXPORT int apc_recurrent_step_bf16(const void* x, int ldx, const void* y, int ldy, const float* in_bias, const float* conv_w,
                                       const float* conv_b, int taps, float* conv_state, const void* W, const float* zb, int parts,
                                       const float* rate, const float* yb, float out_scale, float* state, int M, int C,
                                       const int* row_seg, const int* conv_slots, const int* slots, void* out, int ldo,
                                       hipStream_t stream) {
  if (M <= 0) return 0;
  if (!apc_recurrent_step_bf16_takes(M, C, parts, taps, ldx, ldy, ldo)) return APC_ERR_UNSUPPORTED;
  if (!x || !y || !conv_w || !conv_state || !W || !zb || !rate || !state || !row_seg || !conv_slots || !slots || !out || ldx < C ||
      ldy < C || ldo < C || (((uintptr_t)x | (uintptr_t)W | (uintptr_t)conv_state | (uintptr_t)state | (uintptr_t)zb | (uintptr_t)rate |
      (uintptr_t)yb) & 15u) || (((uintptr_t)y | (uintptr_t)out) & 7u))
    return APC_ERR_BAD_ARG;
  const StepArgs A{(const bf16_t*)x, (const bf16_t*)y, ldx, ldy, in_bias, conv_w, conv_b, conv_state, (const bf16_t*)W, zb, rate, yb,
                   out_scale, state, row_seg, conv_slots, slots, (bf16_t*)out, ldo, M, C, C / parts};
#define STEP_LAUNCH(TAPS_, CHUNKS_) \
  hipLaunchKernelGGL((recurrent_step_kernel<TAPS_, CHUNKS_>), dim3(parts), dim3(STEP_WAVES * 64), 0, stream, A)
#define STEP_BY_W(TAPS_)                                                                                          \
  switch (A.w) {                                                                                                  \
    case 32: STEP_LAUNCH(TAPS_, 1); break;                                                                        \
    case 64: STEP_LAUNCH(TAPS_, 2); break;                                                                        \
    case 128: STEP_LAUNCH(TAPS_, 4); break;                                                                       \
    default: STEP_LAUNCH(TAPS_, 8); break;                                                                        \
  }
  if (taps == 2) { STEP_BY_W(2) } else if (taps == 3) { STEP_BY_W(3) } else { STEP_BY_W(4) }
#undef STEP_BY_W
#undef STEP_LAUNCH
  APC_LAUNCH_CHECK();
  return 0;
}
