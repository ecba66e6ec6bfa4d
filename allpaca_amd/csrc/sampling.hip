// Token choice on the GPU: first-maximum argmax, and temperature / top-k / top-p
// sampling with a uniform number given per row.  Two ways to the same tokens: one block
// per row of logits (thresholds by bisection; needs no working memory), and, for rows as
// long as a real vocabulary, many blocks a row with thresholds by radix descent (second
// half of this file).
//
// Semantics follow crates/allpaca-core/src/sampling.rs:24-67, 215-331:
//   all logits non-finite -> token 0;  temperature <= 1e-5 -> argmax (first maximum);
//   else v = logit / max(T, 1e-5) for finite logits;  top-k keeps the k largest in
//   the order (v descending, id ascending);  top-p (0 <= p < 1) keeps the shortest
//   prefix of that order whose probability (over what top-k left) reaches p;
//   softmax over the survivors;  the draw walks r -= p_i until r <= 0, in sorted
//   order if top-k or top-p cut or sorted the list, else in id order.
// The random number is an input, so a token depends on (seed, request, position)
// only, never on the batch.
#include "common.h"
#include "no_alloc.h"
#include <math.h>
#include <algorithm>
#include <string.h>
#include <mutex>

constexpr int SNT = 256;
constexpr int SMALL_MAX = 1024;  // survivors of top-k handled in LDS in the reference's own sequential order

__device__ __forceinline__ uint32_t key_of(float v) {  // monotone map; 0 is reserved for "not a candidate"
  const uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float value_of(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ bool finite_f(float v) { return fabsf(v) <= 3.402823466e+38f; }  // false for NaN, inf

struct Cut {  // the set { key > tau  or  (key == tau and id <= id_cut) }
  uint32_t tau;
  int id_cut;
};
__device__ __forceinline__ bool in_cut(const Cut& c, uint32_t key, int id) {
  return key > c.tau || (key == c.tau && id <= c.id_cut);
}

template <typename T>
__device__ __forceinline__ T block_sum_t(T v, T* smem) {
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
  __syncthreads();
  if (threadIdx.x % WAVE == 0) smem[threadIdx.x / WAVE] = v;
  __syncthreads();
  T t = smem[0];
#pragma unroll
  for (int i = 1; i < SNT / WAVE; ++i) t += smem[i];
  return t;
}

struct RowView {
  const float* logits;
  int V;
  float inv_t;  // scaled value = logit / t, computed as a division to match the reference
  float t;
  __device__ __forceinline__ uint32_t key(int i) const {
    const float x = logits[i];
    return finite_f(x) ? key_of(x / t) : 0u;
  }
};

// number of elements of `set` with key >= trial
__device__ uint32_t count_ge(const RowView& rv, const Cut& set, uint32_t trial, uint32_t* smem) {
  uint32_t c = 0;
  for (int i = threadIdx.x; i < rv.V; i += SNT) {
    const uint32_t k = rv.key(i);
    c += (k != 0u && k >= trial && in_cut(set, k, i)) ? 1u : 0u;
  }
  return block_sum_t<uint32_t>(c, smem);
}
// number of elements of `set` with key == tau and id < id_trial
__device__ uint32_t count_eq_below(const RowView& rv, const Cut& set, uint32_t tau, int id_trial, uint32_t* smem) {
  uint32_t c = 0;
  for (int i = threadIdx.x; i < rv.V && i < id_trial; i += SNT) {
    const uint32_t k = rv.key(i);
    c += (k == tau && in_cut(set, k, i)) ? 1u : 0u;
  }
  return block_sum_t<uint32_t>(c, smem);
}
// mass = sum exp(v - vmax) over elements of `set` with key >= trial
__device__ float mass_ge(const RowView& rv, const Cut& set, uint32_t trial, float vmax, float* smem) {
  float s = 0.f;
  for (int i = threadIdx.x; i < rv.V; i += SNT) {
    const uint32_t k = rv.key(i);
    if (k != 0u && k >= trial && in_cut(set, k, i)) s += expf(value_of(k) - vmax);
  }
  return block_sum_t<float>(s, smem);
}

// the `need`-th (1-based) smallest id among elements of `set` with key == tau
__device__ int nth_tie(const RowView& rv, const Cut& set, uint32_t tau, uint32_t need, uint32_t* smem) {
  int id = 0;
  int top = 1;
  while (top < rv.V) top <<= 1;
  for (int bit = top; bit > 0; bit >>= 1) {
    const int trial = id | bit;
    if (count_eq_below(rv, set, tau, trial, smem) < need) id = trial;
  }
  return id;
}

// the k largest elements of `set` (|set| >= k >= 1) in (key desc, id asc) order
__device__ Cut select_by_count(const RowView& rv, const Cut& set, uint32_t k, uint32_t* smem) {
  uint32_t tau = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t trial = tau | (1u << bit);
    if (count_ge(rv, set, trial, smem) >= k) tau = trial;
  }
  const uint32_t c_ge = count_ge(rv, set, tau, smem);
  const uint32_t c_gt = (tau == 0xffffffffu) ? 0u : count_ge(rv, set, tau + 1u, smem);
  Cut out;
  out.tau = tau;
  if (c_ge <= k) { out.id_cut = set.tau == tau ? set.id_cut : 0x7fffffff; return out; }
  out.id_cut = nth_tie(rv, set, tau, k - c_gt, smem);
  return out;
}

// the shortest prefix of `set` in sorted order whose mass reaches `target`; *reached = false if none does
__device__ Cut select_by_mass(const RowView& rv, const Cut& set, float target, float vmax, bool* reached, float* fsm,
                              uint32_t* usm) {
  const uint32_t lowest = set.tau == 0u ? 1u : set.tau;
  if (!(mass_ge(rv, set, lowest, vmax, fsm) >= target)) { *reached = false; return set; }
  *reached = true;
  uint32_t tau = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t trial = tau | (1u << bit);
    const float ms = mass_ge(rv, set, trial, vmax, fsm);
    if (ms >= target && ms > 0.f) tau = trial;  // ms > 0 keeps tau on an element when target <= 0
  }
  if (tau < lowest) tau = lowest;
  const float m_gt = (tau == 0xffffffffu) ? 0.f : mass_ge(rv, set, tau + 1u, vmax, fsm);
  const uint32_t c_eq = count_ge(rv, set, tau, usm) - ((tau == 0xffffffffu) ? 0u : count_ge(rv, set, tau + 1u, usm));
  const float p_tau = expf(value_of(tau) - vmax);
  uint32_t need = 1;
  if (p_tau > 0.f) {
    const float n = ceilf((target - m_gt) / p_tau);
    need = n < 1.f ? 1u : (n > (float)c_eq ? c_eq : (uint32_t)n);
  }
  if (need < 1u) need = 1u;
  Cut out;
  out.tau = tau;
  out.id_cut = nth_tie(rv, set, tau, need, usm);
  return out;
}

__global__ __launch_bounds__(SNT) void argmax_rows_kernel(const float* __restrict__ logits, int ldl, int V,
                                                          int* __restrict__ out) {
  __shared__ float bv[SNT / WAVE];
  __shared__ int bi[SNT / WAVE];
  const float* row = logits + (size_t)blockIdx.x * ldl;
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  for (int i = threadIdx.x; i < V; i += SNT) {
    const float v = row[i];
    if (v > best) { best = v; best_i = i; }  // strict: the first maximum of this thread's ascending ids
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, WAVE);
    const int oi = __shfl_xor(best_i, o, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
  }
  if (threadIdx.x % WAVE == 0) { bv[threadIdx.x / WAVE] = best; bi[threadIdx.x / WAVE] = best_i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SNT / WAVE; ++w)
      if (bv[w] > best || (bv[w] == best && bi[w] < best_i)) { best = bv[w]; best_i = bi[w]; }
    out[blockIdx.x] = best_i == 0x7fffffff ? 0 : best_i;  // nothing above -inf: token 0 (sampling.rs:215-225)
  }
}

// Wide rows are cut into pieces so that more than one block works on a row: a first pass leaves the first
// maximum of every piece (value, id), a second pass takes the first maximum of those.
__global__ __launch_bounds__(SNT) void argmax_pieces_kernel(const float* __restrict__ logits, int ldl, int V, int piece,
                                                            float* __restrict__ pv, int* __restrict__ pi) {
  __shared__ float bv[SNT / WAVE];
  __shared__ int bi[SNT / WAVE];
  const float* row = logits + (size_t)blockIdx.x * ldl;
  const int lo = blockIdx.y * piece, hi = min(V, lo + piece);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  for (int i = lo + threadIdx.x; i < hi; i += SNT) {
    const float v = row[i];
    if (v > best) { best = v; best_i = i; }
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, WAVE);
    const int oi = __shfl_xor(best_i, o, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
  }
  if (threadIdx.x % WAVE == 0) { bv[threadIdx.x / WAVE] = best; bi[threadIdx.x / WAVE] = best_i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SNT / WAVE; ++w)
      if (bv[w] > best || (bv[w] == best && bi[w] < best_i)) { best = bv[w]; best_i = bi[w]; }
    pv[(size_t)blockIdx.x * gridDim.y + blockIdx.y] = best;
    pi[(size_t)blockIdx.x * gridDim.y + blockIdx.y] = best_i;
  }
}

__global__ __launch_bounds__(WAVE) void argmax_final_kernel(const float* __restrict__ pv, const int* __restrict__ pi,
                                                            int pieces, int* __restrict__ out) {
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  for (int p = threadIdx.x; p < pieces; p += WAVE) {
    const float v = pv[(size_t)blockIdx.x * pieces + p];
    const int i = pi[(size_t)blockIdx.x * pieces + p];
    if (v > best || (v == best && i < best_i)) { best = v; best_i = i; }
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, WAVE);
    const int oi = __shfl_xor(best_i, o, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
  }
  if (threadIdx.x == 0) out[blockIdx.x] = best_i == 0x7fffffff ? 0 : best_i;
}

// `scratch`: room for 2 * n_rows * 64 four-byte values, or null for the one-pass kernel
APC_EXPORT int apc_argmax_rows(const float* logits, int ldl, int n_rows, int V, int* out, void* scratch,
                               hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (V <= 0 || ldl < V) return APC_ERR_BAD_ARG;
  if (!scratch || V < 8192 || n_rows > 65535) {
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(n_rows), dim3(SNT), 0, stream, logits, ldl, V, out);
    APC_LAUNCH_CHECK();
    return 0;
  }
  const int pieces = 64;
  const int piece = ceil_div(V, pieces);
  float* pv = (float*)scratch;
  int* pi = (int*)scratch + (size_t)n_rows * pieces;
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(n_rows, pieces), dim3(SNT), 0, stream, logits, ldl, V, piece, pv, pi);
  APC_LAUNCH_CHECK();
  hipLaunchKernelGGL(argmax_final_kernel, dim3(n_rows), dim3(WAVE), 0, stream, pv, pi, pieces, out);
  APC_LAUNCH_CHECK();
  return 0;
}

// ---- the variant that allocates nothing (declared in no_alloc.h) ----
// Room for the pieces of APC_ARGMAX_NO_ALLOC_MAX_ROWS rows: values [rows][64], then indices [rows][64].  Each GPU holds
// its own copy of the array at its own address; in host code the array's name is not that address, so the address is
// asked for once per device (hipGetSymbolAddress, with that device current) and only the answer is handed to kernels.
constexpr int NO_ALLOC_PIECES = 64;
static __device__ __align__(256) unsigned char argmax_scratch[(size_t)APC_ARGMAX_NO_ALLOC_MAX_ROWS * NO_ALLOC_PIECES * 8];
constexpr int NO_ALLOC_MAX_DEVICES = 64;
static void* argmax_scratch_ptr[NO_ALLOC_MAX_DEVICES];  // per device, null until its first call
static std::mutex argmax_scratch_lock;

APC_EXPORT int apc_argmax_rows_no_alloc(const float* logits, int ldl, int n_rows, int V, int* out,
                                        hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (V <= 0 || ldl < V || !logits || !out) return APC_ERR_BAD_ARG;
  if (n_rows > APC_ARGMAX_NO_ALLOC_MAX_ROWS) return APC_ERR_TOO_LARGE;
  if (V < 8192) {  // one block a row: no pieces, nothing beyond input and output
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(n_rows), dim3(SNT), 0, stream, logits, ldl, V, out);
    APC_LAUNCH_CHECK();
    return 0;
  }
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= NO_ALLOC_MAX_DEVICES) return APC_ERR_UNSUPPORTED;
  void* ptr;
  {
    std::lock_guard<std::mutex> hold(argmax_scratch_lock);
    if (!argmax_scratch_ptr[dev]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(argmax_scratch));
      if (e != hipSuccess) return (int)e;
      if (!p) return (int)hipErrorInvalidSymbol;
      argmax_scratch_ptr[dev] = p;
    }
    ptr = argmax_scratch_ptr[dev];
  }
  const int piece = ceil_div(V, NO_ALLOC_PIECES);
  float* pv = (float*)ptr;
  int* pi = (int*)ptr + (size_t)n_rows * NO_ALLOC_PIECES;
  hipLaunchKernelGGL(argmax_pieces_kernel, dim3(n_rows, NO_ALLOC_PIECES), dim3(SNT), 0, stream, logits, ldl, V, piece,
                     pv, pi);
  APC_LAUNCH_CHECK();
  hipLaunchKernelGGL(argmax_final_kernel, dim3(n_rows), dim3(WAVE), 0, stream, pv, pi, NO_ALLOC_PIECES, out);
  APC_LAUNCH_CHECK();
  return 0;
}

// What a block's threads share while they choose one row's token
struct alignas(16) SampleShared {
  float fsm[SNT / WAVE];
  uint32_t usm[SNT / WAVE];
  float bv[SNT / WAVE];
  int bi[SNT / WAVE];
  uint32_t s_key[SMALL_MAX], s_key2[SMALL_MAX];
  int s_id[SMALL_MAX], s_id2[SMALL_MAX];
  uint32_t s_count;
  int s_answer;
};

// The few survivors of a cut (cnt of them, in sh.s_key / sh.s_id in any order): sorted by (value descending, id
// ascending), then one thread does the reference's sequential arithmetic.
__device__ __forceinline__ void sample_few(SampleShared& sh, int cnt, bool use_top_p, float tp, float r, int* out_row) {
  uint32_t* s_key = sh.s_key; uint32_t* s_key2 = sh.s_key2;
  int* s_id = sh.s_id; int* s_id2 = sh.s_id2;
  for (int e = threadIdx.x; e < cnt; e += SNT) {
    const uint32_t k = s_key[e];
    const int id = s_id[e];
    int rank = 0;
    for (int j = 0; j < cnt; ++j) rank += (s_key[j] > k || (s_key[j] == k && s_id[j] < id)) ? 1 : 0;
    s_key2[rank] = k;
    s_id2[rank] = id;
  }
  __syncthreads();
  // the exponentials by all threads (the unsorted keys are done with: their place holds them), the sums by one
  float* e = reinterpret_cast<float*>(s_key);
  const float vmax = value_of(s_key2[0]);
  for (int i = threadIdx.x; i < cnt; i += SNT) e[i] = expf(value_of(s_key2[i]) - vmax);
  __syncthreads();
  if (threadIdx.x == 0) {
    int m = cnt;
    if (use_top_p) {
      float sum = 0.f;
      for (int i = 0; i < m; ++i) sum += e[i];
      if (sum == 0.f || !finite_f(sum)) {
        int keep = (int)ceilf(tp * (float)m);
        m = keep < 1 ? 1 : (keep > m ? m : keep);
      } else {
        float acc = 0.f;
        for (int i = 0; i < m; ++i) {
          acc += e[i] / sum;
          if (acc >= tp) { m = i + 1; break; }
        }
      }
    }
    float sum = 0.f;
    for (int i = 0; i < m; ++i) sum += e[i];
    float rr = r;
    int pick = s_id2[m - 1];
    for (int i = 0; i < m; ++i) {
      const float p = sum == 0.f ? 1.0f / (float)m : e[i] / sum;
      rr -= p;
      if (rr <= 0.f) { pick = s_id2[i]; break; }
    }
    *out_row = pick;
  }
}

// One row by one block, every step a pass of the block over the whole row (thresholds by bisection): the way for
// callers without working memory, and for rows that the kernels below hand back.
__device__ __forceinline__ void sample_row_one_block(SampleShared& sh, const float* __restrict__ lg, int V, float T,
                                                     int tk, float tp, float r, int* out_row) {
  float* fsm = sh.fsm; uint32_t* usm = sh.usm; float* bv = sh.bv; int* bi = sh.bi;
  uint32_t* s_key = sh.s_key; int* s_id = sh.s_id;
  uint32_t& s_count = sh.s_count; int& s_answer = sh.s_answer;

  // pass 1: argmax of the raw logits (first maximum) and the number of finite ones
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t nfin = 0;
  for (int i = threadIdx.x; i < V; i += SNT) {
    const float v = lg[i];
    if (v > best) { best = v; best_i = i; }
    nfin += finite_f(v) ? 1u : 0u;
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, WAVE);
    const int oi = __shfl_xor(best_i, o, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
  }
  if (threadIdx.x % WAVE == 0) { bv[threadIdx.x / WAVE] = best; bi[threadIdx.x / WAVE] = best_i; }
  __syncthreads();
  for (int w = 0; w < SNT / WAVE; ++w)
    if (bv[w] > best || (bv[w] == best && bi[w] < best_i)) { best = bv[w]; best_i = bi[w]; }
  const int arg = best_i == 0x7fffffff ? 0 : best_i;
  nfin = block_sum_t<uint32_t>(nfin, usm);

  if (nfin == 0u) { if (threadIdx.x == 0) *out_row = 0; return; }
  if (T <= 1e-5f) { if (threadIdx.x == 0) *out_row = arg; return; }

  RowView rv;
  rv.logits = lg;
  rv.V = V;
  rv.t = fmaxf(T, 1e-5f);
  rv.inv_t = 1.0f / rv.t;

  Cut set;  // all finite logits
  set.tau = 0u;
  set.id_cut = -1;
  uint32_t n = nfin;
  bool sorted = false;
  if (tk > 0 && n > (uint32_t)tk) {
    set = select_by_count(rv, set, (uint32_t)tk, usm);
    n = (uint32_t)tk;
    sorted = true;
  }
  const bool use_top_p = tp >= 0.0f && tp < 1.0f && n > 1u;

  if (n <= (uint32_t)SMALL_MAX && (sorted || use_top_p)) {
    // few survivors: gather, sort, then one thread does the reference's sequential arithmetic
    if (threadIdx.x == 0) s_count = 0u;
    __syncthreads();
    for (int i = threadIdx.x; i < V; i += SNT) {
      const uint32_t k = rv.key(i);
      if (k != 0u && in_cut(set, k, i)) {
        const uint32_t at = atomicAdd(&s_count, 1u);
        if (at < (uint32_t)SMALL_MAX) { s_key[at] = k; s_id[at] = i; }
      }
    }
    __syncthreads();
    const int cnt = (int)min(s_count, (uint32_t)SMALL_MAX);
    sample_few(sh, cnt, use_top_p, tp, r, out_row);
    return;
  }

  // many survivors: thresholds found by bisection on the key, sums by block reductions
  const float vmax = best / rv.t;  // the largest finite scaled logit (best is finite here unless +inf is present)
  float vmax_f = vmax;
  if (!finite_f(best)) {           // +inf among the logits: take the largest finite one instead
    float fm = -INFINITY;
    for (int i = threadIdx.x; i < V; i += SNT) { const float v = lg[i]; if (finite_f(v)) fm = fmaxf(fm, v); }
    fm = block_max<SNT>(fm, fsm);
    vmax_f = fm / rv.t;
  }
  if (use_top_p) {
    const uint32_t lowest = set.tau == 0u ? 1u : set.tau;
    const float total = mass_ge(rv, set, lowest, vmax_f, fsm);
    if (total == 0.f || !finite_f(total)) {
      const int keep = (int)ceilf(tp * (float)n);
      const uint32_t kk = (uint32_t)(keep < 1 ? 1 : (keep > (int)n ? (int)n : keep));
      set = select_by_count(rv, set, kk, usm);
    } else {
      bool reached;
      const Cut c = select_by_mass(rv, set, tp * total, vmax_f, &reached, fsm, usm);
      if (reached) set = c;
    }
    sorted = true;
  }
  const uint32_t lowest = set.tau == 0u ? 1u : set.tau;
  const float total = mass_ge(rv, set, lowest, vmax_f, fsm);
  const float target = r * total;
  if (sorted) {
    bool reached;
    const Cut c = select_by_mass(rv, set, target, vmax_f, &reached, fsm, usm);
    if (reached) { if (threadIdx.x == 0) *out_row = c.id_cut; return; }
    // rounding left r above the whole mass: the last candidate in sorted order
    uint32_t kmin = 0xffffffffu;
    for (int i = threadIdx.x; i < V; i += SNT) {
      const uint32_t k = rv.key(i);
      if (k != 0u && in_cut(set, k, i)) kmin = min(kmin, k);
    }
    // min over the block through the float-free path: reuse count_ge by bisection is overkill; do an LDS min
    __syncthreads();
    if (threadIdx.x == 0) s_count = 0xffffffffu;
    __syncthreads();
    atomicMin(&s_count, kmin);
    __syncthreads();
    kmin = s_count;
    int imax = -1;
    for (int i = threadIdx.x; i < V; i += SNT) {
      const uint32_t k = rv.key(i);
      if (k == kmin && in_cut(set, k, i)) imax = max(imax, i);
    }
    __syncthreads();
    if (threadIdx.x == 0) s_answer = -1;
    __syncthreads();
    atomicMax(&s_answer, imax);
    __syncthreads();
    if (threadIdx.x == 0) *out_row = s_answer < 0 ? 0 : s_answer;
    return;
  }
  // id order: the first id whose running mass reaches the target
  if (threadIdx.x == 0) s_answer = -1;
  __syncthreads();
  float running = 0.f;
  int last_in = -1;
  for (int base = 0; base < V; base += SNT) {
    const int i = base + threadIdx.x;
    float e = 0.f;
    bool in = false;
    if (i < V) {
      const uint32_t k = rv.key(i);
      in = k != 0u && in_cut(set, k, i);
      if (in) { e = expf(value_of(k) - vmax_f); last_in = i; }
    }
    // inclusive scan over the block in id order
    float s = e;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const float up = __shfl_up(s, o, WAVE);
      if ((threadIdx.x % WAVE) >= o) s += up;
    }
    __syncthreads();
    if (threadIdx.x % WAVE == WAVE - 1) fsm[threadIdx.x / WAVE] = s;
    __syncthreads();
    float before = running;
    for (int w = 0; w < threadIdx.x / WAVE; ++w) before += fsm[w];
    float chunk = 0.f;
    for (int w = 0; w < SNT / WAVE; ++w) chunk += fsm[w];
    const float cum = before + s;
    if (in && cum >= target) atomicMin((unsigned int*)&s_answer, (unsigned int)i);  // -1 is the largest unsigned
    running += chunk;
    __syncthreads();
    if (s_answer >= 0) break;
  }
  if (s_answer < 0) {  // r above the whole mass by rounding: the last candidate
    __syncthreads();
    if (threadIdx.x == 0) s_count = 0u;
    __syncthreads();
    if (last_in >= 0) atomicMax(&s_count, (uint32_t)last_in);
    __syncthreads();
    if (threadIdx.x == 0) *out_row = (int)s_count;
    return;
  }
  if (threadIdx.x == 0) *out_row = s_answer;
}

__global__ __launch_bounds__(SNT) void sample_rows_kernel(const float* __restrict__ logits, int ldl, int V,
                                                          const float* __restrict__ temperature,
                                                          const int* __restrict__ top_k,
                                                          const float* __restrict__ top_p,
                                                          const float* __restrict__ uniform, int* __restrict__ out) {
  __shared__ SampleShared sh;
  const int row = blockIdx.x;
  sample_row_one_block(sh, logits + (size_t)row * ldl, V, temperature[row], top_k[row], top_p[row], uniform[row],
                       out + row);
}

// ---- The same rules with many blocks a row ----
// A row of a real vocabulary is half a megabyte, and one block's passes over it (about a hundred of them for top-p)
// took 4-17 ms.  Here every step is one launch over (pieces of a row) x (rows), and the thresholds come from radix
// descents instead of bisection.  The candidates stand in one order, by (value descending, id ascending), written as
// one 64-bit sort key (the value's key, then the id counted down); the candidate at which a running weight first
// reaches a target is found digit by digit, 13 bits at a time, from a histogram of the weights per digit value: four
// launches a threshold for vocabularies up to a million, and equal values need no special case.  The weights are
// integers (1 for top-k; for probabilities exp(v - vmax) in units of 2^-40, at least 1), so that sums do not depend
// on the order in which blocks and threads add them: a row's token is the same whatever the batch and the grid.
// Launches, each of which a row sits out if it has no use for it:  the maximum;  top-k: 4;  top-p: 4;  the draw: 4
// (a list that no cut has sorted is walked in id order: the sort key is then the id alone);  the end, which writes the
// tokens.  What one launch finds the next one reads: every block of a row first works out, from the histogram of
// the launch before, where the row stands (the same arithmetic in each of them), then adds its piece of the row to
// the next histogram.  A histogram has two levels (8,192 values and their sums in groups of 32), so that a block
// reads 256 + 32 numbers of it, not all.
// Few survivors (up to SMALL_MAX after top-k) are gathered and go through the reference's sequential arithmetic as
// above.
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

typedef unsigned long long u64;
constexpr int PNT = 1024;                // threads of a block that works on a piece of a row
constexpr int DIGIT_BITS = 13;
constexpr int FINE = 1 << DIGIT_BITS;    // digit values
constexpr int GROUP = 8;                 // digit values a group
constexpr int COARSE = FINE / GROUP;     // groups
static_assert(COARSE == PNT, "a thread adds one group");
constexpr int MAX_PIECES = 32;
constexpr int N_SELECTS = 3;             // top-k, top-p, the draw
constexpr int MAX_DIGITS = 5;            // 64 bits of sort key
constexpr int ROTA = 3;                  // histograms in use in turn: written, read, cleared
constexpr float MASS_ONE = 0x1p40f;      // weight of the row's largest value

enum { ST_TOPK = 0, ST_TOPP = 1, ST_DRAW = 2 };
enum { PH_ACTIVE = 1, PH_FEW = 2, PH_DONE = 3, PH_ONE_BLOCK = 4 };
enum { SEEN_TOPK = 1, SEEN_TOPP = 2 };

// digit d is bits [digit_lo, digit_hi) of the sort key
__host__ __device__ constexpr int digit_hi(int d) { return 64 - DIGIT_BITS * d; }
__host__ __device__ constexpr int digit_lo(int d) { return digit_hi(d) > DIGIT_BITS ? digit_hi(d) - DIGIT_BITS : 0; }

struct RowState {
  int phase, result;
  float t, vmax;           // temperature in use, the largest finite scaled value
  uint32_t n;              // candidates left
  int sorted;              // a cut has put the list in sorted order
  uint32_t set_tau;        // the candidates: key > set_tau, or key == set_tau and id <= set_id
  int set_id;
  int descending;          // the launch before left a histogram of this row
  int by_id;               // ... ordered by id (the draw from an unsorted list)
  int seen;                // cuts this row has passed
  int pad;
  u64 prefix;              // digits found so far
  u64 above;               // weight in front of the prefix
  u64 target;              // the threshold stands at the first candidate with this much weight up to and including it
  u64 total;
};

// Sizes of a call: what the kernels need to know of the row and of its sort key
struct SampleShape {
  int ldl, V, R, chunk, pieces;
  int vec;                 // rows start at multiples of 16 bytes: four values a load
  int id_bits;             // bits of an id
  int key_digits;          // digits of a sort key by (value, id)
  int id_digits;           // ... by id alone
};

// The rows' options: on the device, or, of up to BY_VALUE rows, with the launch (no copy to the device in front of it).
constexpr int BY_VALUE = 64;
struct RowOptions { const float *temperature, *top_p, *uniform; const int* top_k; };
struct RowValues { float temperature[BY_VALUE], top_p[BY_VALUE], uniform[BY_VALUE]; int top_k[BY_VALUE]; };

struct SampleSpace {
  u64* fine;               // [ROTA][row][FINE]
  u64* coarse;             // [ROTA][row][COARSE]
  uint32_t* few_count;     // [row]
  float* piece_best;       // [row][MAX_PIECES] ...
  int* piece_arg;
  uint32_t* piece_finite;
  float* piece_finite_max;
  RowState* state;         // [launch + 1][row]
  uint32_t* few_key;       // [row][SMALL_MAX]
  int* few_id;
  RowValues* options;      // where options that came with the first launch stand for the others
  size_t bytes;
};

constexpr size_t round16(size_t n) { return (n + 15) / 16 * 16; }

SampleSpace carve(void* base, int R) {
  SampleSpace s;
  size_t at = 0;
  auto take = [&](size_t bytes) { char* q = (char*)((uintptr_t)base + at); at += round16(bytes); return q; };
  const size_t r = (size_t)R;
  s.fine = (u64*)take(ROTA * r * FINE * sizeof(u64));
  s.coarse = (u64*)take(ROTA * r * COARSE * sizeof(u64));
  s.few_count = (uint32_t*)take(r * 4);
  s.piece_best = (float*)take(r * MAX_PIECES * 4);
  s.piece_arg = (int*)take(r * MAX_PIECES * 4);
  s.piece_finite = (uint32_t*)take(r * MAX_PIECES * 4);
  s.piece_finite_max = (float*)take(r * MAX_PIECES * 4);
  s.state = (RowState*)take((N_SELECTS * MAX_DIGITS + 1) * r * sizeof(RowState));
  s.few_key = (uint32_t*)take(r * SMALL_MAX * 4);
  s.few_id = (int*)take(r * SMALL_MAX * 4);
  s.options = (RowValues*)take(sizeof(RowValues));
  s.bytes = at;
  return s;
}

// pieces of a row: enough blocks for the chip when the rows are few, at least 4 values a thread
void cut_row(int R, int V, int* pieces, int* chunk) {
  int want = ceil_div(512, R);
  want = want > MAX_PIECES ? MAX_PIECES : want;
  const int most = ceil_div(V, 4 * PNT);
  *pieces = want < most ? want : most;
  *chunk = ceil_div(ceil_div(V, *pieces), 4) * 4;
  *pieces = ceil_div(V, *chunk);
}

// f(i, logits[i]) for the values i0 <= i < i1 of a row, a thread's values in ascending order
template <typename F>
__device__ __forceinline__ void for_piece(const float* __restrict__ lg, int vec, int i0, int i1, F&& f) {
  if (vec) {  // i0 is a multiple of 4
    for (int i = i0 + 4 * (int)threadIdx.x; i < i1; i += 4 * PNT) {
      if (i + 3 < i1) {
        const float4 x = *reinterpret_cast<const float4*>(lg + i);
        f(i, x.x);
        f(i + 1, x.y);
        f(i + 2, x.z);
        f(i + 3, x.w);
      } else {
        for (int j = i; j < i1; ++j) f(j, lg[j]);
      }
    }
  } else {
    for (int i = i0 + (int)threadIdx.x; i < i1; i += PNT) f(i, lg[i]);
  }
}

// inclusive sums over the block's NT threads in thread order, and the sum of all
template <int NT>
__device__ __forceinline__ u64 block_scan(u64 v, u64* total, u64* smem) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const u64 up = __shfl_up(v, o, WAVE);
    if (lane >= o) v += up;
  }
  __syncthreads();
  if (lane == WAVE - 1) smem[wave] = v;
  __syncthreads();
  u64 before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / WAVE; ++w) {
    const u64 x = smem[w];
    all += x;
    if (w < wave) before += x;
  }
  *total = all;
  return v + before;
}

// The sort key: larger = earlier.  The id part counts down and stands in the top bits of its half, so that the
// digits that matter come first; by id alone it stands in the upper half.
__device__ __forceinline__ u64 sort_key(uint32_t key, int i, int id_bits, int by_id) {
  const uint32_t ik = (((1u << id_bits) - 1u) - (uint32_t)i) << (32 - id_bits);
  return by_id ? ((u64)ik << 32) : (((u64)key << 32) | ik);
}
__device__ __forceinline__ int id_of_sort_key(u64 c, int id_bits, int by_id) {
  const uint32_t ik = by_id ? (uint32_t)(c >> 32) : (uint32_t)c;
  return (int)(((1u << id_bits) - 1u) - (ik >> (32 - id_bits)));
}
__device__ __forceinline__ u64 mass_of(uint32_t key, float vmax) {
  const u64 q = (u64)(expf(value_of(key) - vmax) * MASS_ONE);
  return q < 1 ? 1 : q;
}

struct SettleShared {
  u64 scan[PNT / WAVE];
  int bin;
  u64 above;
};

// Where the row stands after launch (stage, digit), whose histogram is (fine, coarse): all NT threads of the block,
// the same result in each.
template <int NT>
__device__ __forceinline__ void settle(RowState& S, const SampleShape& sz, int stage, int digit,
                                       const u64* __restrict__ fine, const u64* __restrict__ coarse, float frac,
                                       SettleShared& sh) {
  if (S.phase != PH_ACTIVE || !S.descending) return;
  constexpr int PER = COARSE / NT;  // groups a thread, threads in descending order of the digit's value
  const int top = COARSE - 1 - threadIdx.x * PER;
  u64 groups[PER], local = 0;
#pragma unroll
  for (int g = 0; g < PER; ++g) {
    groups[g] = coarse[top - g];
    local += groups[g];
  }
  if (threadIdx.x == 0) sh.bin = -1;
  u64 all;
  const u64 incl = block_scan<NT>(local, &all, sh.scan);
  if (digit == 0 && stage != ST_TOPK) {  // every candidate is in this histogram: the threshold as a weight
    S.total = all;
    const double want = ceil((double)frac * (double)all);
    const u64 target = want <= 1.0 ? 1 : (want >= (double)all ? all : (u64)want);
    S.target = target > all ? all : target;
  }
  u64 before = S.above + incl - local;
  if (before < S.target && S.target <= before + local) {
#pragma unroll
    for (int g = 0; g < PER; ++g) {
      if (before < S.target && S.target <= before + groups[g]) {
        u64 mine[GROUP];
#pragma unroll
        for (int k = 0; k < GROUP; ++k) mine[k] = fine[(top - g) * GROUP + GROUP - 1 - k];
        u64 at = before;
#pragma unroll
        for (int k = 0; k < GROUP; ++k) {
          if (at < S.target && S.target <= at + mine[k]) {
            sh.bin = (top - g) * GROUP + GROUP - 1 - k;
            sh.above = at;
          }
          at += mine[k];
        }
      }
      before += groups[g];
    }
  }
  __syncthreads();
  const int bin = sh.bin;
  const u64 above = sh.above;
  __syncthreads();
  if (bin < 0) {  // the weight asked for is not there (it always is): the one-block way decides
    S.phase = PH_ONE_BLOCK;
    return;
  }
  S.prefix |= (u64)bin << digit_lo(digit);
  S.above = above;
  if (digit < (S.by_id ? sz.id_digits : sz.key_digits) - 1) return;
  // the sort key is whole: it names one candidate
  S.descending = 0;
  const int id = id_of_sort_key(S.prefix, sz.id_bits, S.by_id);
  if (stage == ST_DRAW) {
    S.phase = PH_DONE;
    S.result = id;
    return;
  }
  S.set_tau = (uint32_t)(S.prefix >> 32);
  S.set_id = id;
  S.sorted = 1;
  if (stage == ST_TOPK) S.n = (uint32_t)S.target;
}

// RowValues: the rows' options came with this launch and are put where the later ones look for them.
struct NoValues {};
template <typename Values>
__global__ __launch_bounds__(PNT) void sample_max_kernel(const float* __restrict__ logits, SampleShape sz, Values values, SampleSpace sp) {
  __shared__ float bv[PNT / WAVE], fv[PNT / WAVE];
  __shared__ int bi[PNT / WAVE];
  __shared__ uint32_t nv[PNT / WAVE];
  const int row = blockIdx.y, piece = blockIdx.x;
  // what the first of the later launches adds to (each of them clears the histogram of the one after it)
  for (int j = piece * PNT + threadIdx.x; j < FINE; j += sz.pieces * PNT) sp.fine[(size_t)row * FINE + j] = 0;
  if (piece == 0) {
    sp.coarse[(size_t)row * COARSE + threadIdx.x] = 0;
    if (threadIdx.x == 0) {
      sp.few_count[row] = 0u;
      if constexpr (!__is_same(Values, NoValues)) {
        sp.options->temperature[row] = values.temperature[row];
        sp.options->top_p[row] = values.top_p[row];
        sp.options->uniform[row] = values.uniform[row];
        sp.options->top_k[row] = values.top_k[row];
      }
    }
  }
  const float* lg = logits + (size_t)row * sz.ldl;
  const int i0 = piece * sz.chunk, i1 = min(sz.V, i0 + sz.chunk);
  float best = -INFINITY, fmax = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t nfin = 0;
  for_piece(lg, sz.vec, i0, i1, [&](int i, float v) {
    if (v > best) { best = v; best_i = i; }
    if (finite_f(v)) { ++nfin; fmax = fmaxf(fmax, v); }
  });
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, WAVE);
    const int oi = __shfl_xor(best_i, o, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
    fmax = fmaxf(fmax, __shfl_xor(fmax, o, WAVE));
    nfin += __shfl_xor(nfin, o, WAVE);
  }
  if (threadIdx.x % WAVE == 0) {
    bv[threadIdx.x / WAVE] = best;
    bi[threadIdx.x / WAVE] = best_i;
    fv[threadIdx.x / WAVE] = fmax;
    nv[threadIdx.x / WAVE] = nfin;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < PNT / WAVE; ++w) {
      if (bv[w] > best || (bv[w] == best && bi[w] < best_i)) { best = bv[w]; best_i = bi[w]; }
      fmax = fmaxf(fmax, fv[w]);
      nfin += nv[w];
    }
    const size_t at = (size_t)row * MAX_PIECES + piece;
    sp.piece_best[at] = best;
    sp.piece_arg[at] = best_i;
    sp.piece_finite[at] = nfin;
    sp.piece_finite_max[at] = fmax;
  }
}

struct PassShared {
  u64 hist[FINE];
  SettleShared settle;
};

// Launch `q` of the descents: digit `digit` of `stage`; the one before was (prev_stage, prev_digit), none if q == 0.
__global__ __launch_bounds__(PNT) void sample_pass_kernel(const float* __restrict__ logits, SampleShape sz,
                                                          const float* __restrict__ temperature,
                                                          const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                          const float* __restrict__ uniform, SampleSpace sp, int q,
                                                          int stage, int digit, int prev_stage, int prev_digit) {
  extern __shared__ __attribute__((aligned(16))) unsigned char pass_smem[];
  PassShared& sh = *reinterpret_cast<PassShared*>(pass_smem);
  const int row = blockIdx.y, piece = blockIdx.x, R = sz.R;
  const float* lg = logits + (size_t)row * sz.ldl;
  const float tp = top_p[row];
  const int tk = top_k[row];
  {  // the histogram of the launch after this one
    const size_t next = ((size_t)((q + 1) % ROTA) * R + row);
    for (int j = piece * PNT + threadIdx.x; j < FINE; j += sz.pieces * PNT) sp.fine[next * FINE + j] = 0;
    if (piece == 0) sp.coarse[next * COARSE + threadIdx.x] = 0;
  }
  RowState S;
  if (q == 0) {
    float best = -INFINITY, fmax = -INFINITY;
    int best_i = 0x7fffffff;
    uint32_t nfin = 0;
    for (int p = 0; p < sz.pieces; ++p) {
      const size_t at = (size_t)row * MAX_PIECES + p;
      const float v = sp.piece_best[at];
      const int vi = sp.piece_arg[at];
      if (v > best || (v == best && vi < best_i)) { best = v; best_i = vi; }
      nfin += sp.piece_finite[at];
      fmax = fmaxf(fmax, sp.piece_finite_max[at]);
    }
    const float T = temperature[row];
    S = RowState{};
    S.phase = PH_ACTIVE;
    S.t = fmaxf(T, 1e-5f);
    S.vmax = (finite_f(best) ? best : fmax) / S.t;
    S.n = nfin;
    S.set_tau = 0u;
    S.set_id = -1;
    if (nfin == 0u) { S.phase = PH_DONE; S.result = 0; }
    else if (T <= 1e-5f) { S.phase = PH_DONE; S.result = best_i == 0x7fffffff ? 0 : best_i; }
  } else {
    S = sp.state[(size_t)q * R + row];
    const size_t prev = (size_t)((q - 1) % ROTA) * R + row;
    settle<PNT>(S, sz, prev_stage, prev_digit, sp.fine + prev * FINE, sp.coarse + prev * COARSE,
                prev_stage == ST_TOPP ? tp : uniform[row], sh.settle);
  }
  bool gather = false;
  if (S.phase == PH_ACTIVE && S.descending && digit == 0) S.phase = PH_ONE_BLOCK;  // (the launches of a descent ran out)
  if (S.phase == PH_ACTIVE && !S.descending && digit == 0) {
    auto begin = [&](int by_id, u64 target) {
      S.descending = 1;
      S.by_id = by_id;
      S.prefix = 0;
      S.above = 0;
      S.target = target;
    };
    const bool wants_k = tk > 0 && S.n > (uint32_t)tk && !(S.seen & SEEN_TOPK);
    if (stage == ST_TOPK) {
      if (wants_k) begin(0, (u64)tk);
      S.seen |= SEEN_TOPK;
    } else if (wants_k) {
      S.phase = PH_ONE_BLOCK;          // the caller left out the launches of a cut that this row asks for
    } else {
      const bool use_top_p = tp >= 0.0f && tp < 1.0f && S.n > 1u;
      if (S.n <= (uint32_t)SMALL_MAX && (S.sorted || use_top_p)) {
        S.phase = PH_FEW;
        gather = true;
      } else if (stage == ST_TOPP) {
        if (use_top_p) begin(0, 0);    // the target follows from the sum of this launch's histogram
        S.seen |= SEEN_TOPP;
      } else if (use_top_p && !(S.seen & SEEN_TOPP)) {
        S.phase = PH_ONE_BLOCK;
      } else {
        begin(S.sorted ? 0 : 1, 0);
      }
    }
  }
  if (piece == 0 && threadIdx.x == 0) sp.state[(size_t)(q + 1) * R + row] = S;
  const int i0 = piece * sz.chunk, i1 = min(sz.V, i0 + sz.chunk);
  if (gather) {
    for_piece(lg, sz.vec, i0, i1, [&](int i, float x) {
      if (!finite_f(x)) return;
      const uint32_t k = key_of(x / S.t);
      if (!(k > S.set_tau || (k == S.set_tau && i <= S.set_id))) return;
      const uint32_t at = atomicAdd(&sp.few_count[row], 1u);
      if (at < (uint32_t)SMALL_MAX) {
        sp.few_key[(size_t)row * SMALL_MAX + at] = k;
        sp.few_id[(size_t)row * SMALL_MAX + at] = i;
      }
    });
    return;
  }
  if (S.phase != PH_ACTIVE || !S.descending) return;
#pragma unroll
  for (int k = 0; k < GROUP; ++k) sh.hist[k * PNT + threadIdx.x] = 0;
  __syncthreads();
  const int lo = digit_lo(digit), hi = digit_hi(digit);
  const uint32_t mask = (1u << (hi - lo)) - 1u;
  for_piece(lg, sz.vec, i0, i1, [&](int i, float x) {
    if (!finite_f(x)) return;
    const uint32_t k = key_of(x / S.t);
    if (!(k > S.set_tau || (k == S.set_tau && i <= S.set_id))) return;
    const u64 c = sort_key(k, i, sz.id_bits, S.by_id);
    if (digit > 0 && (c >> hi) != (S.prefix >> hi)) return;
    atomicAdd(&sh.hist[(uint32_t)(c >> lo) & mask], stage == ST_TOPK ? (u64)1 : mass_of(k, S.vmax));
  });
  __syncthreads();
  // thread t adds group t; it starts t values into the group, so that the threads of a wave read different banks
  const size_t cur = (size_t)(q % ROTA) * R + row;
  u64* fine = sp.fine + cur * FINE + threadIdx.x * GROUP;
  u64 sum = 0;
#pragma unroll
  for (int k = 0; k < GROUP; ++k) {
    const int j = (k + threadIdx.x) % GROUP;
    const u64 h = sh.hist[threadIdx.x * GROUP + j];
    if (h) {
      atomicAdd(&fine[j], h);
      sum += h;
    }
  }
  if (sum) atomicAdd(&sp.coarse[cur * COARSE + threadIdx.x], sum);
}

union EndShared {
  SettleShared settle;
  SampleShared one;
};

// The last launch: (last_stage, last_digit) was the one before
__global__ __launch_bounds__(SNT) void sample_end_kernel(const float* __restrict__ logits, SampleShape sz,
                                                         const float* __restrict__ temperature,
                                                         const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                         const float* __restrict__ uniform, SampleSpace sp, int q,
                                                         int last_stage, int last_digit, int* __restrict__ out,
                                                         int* __restrict__ out_host) {
  __shared__ EndShared sh;
  const int row = blockIdx.x, R = sz.R;
  const float tp = top_p[row], r = uniform[row];
  RowState S = sp.state[(size_t)q * R + row];
  const size_t prev = (size_t)((q - 1) % ROTA) * R + row;
  settle<SNT>(S, sz, last_stage, last_digit, sp.fine + prev * FINE, sp.coarse + prev * COARSE,
              last_stage == ST_TOPP ? tp : r, sh.settle);
  if (S.phase == PH_DONE) {
    if (threadIdx.x == 0) {
      out[row] = S.result;
      if (out_host) out_host[row] = S.result;
    }
    return;
  }
  auto to_host = [&]() {                                // (one thread of the block has written out[row])
    __syncthreads();
    if (out_host && threadIdx.x == 0) out_host[row] = *(volatile int*)(out + row);
  };
  __syncthreads();
  if (S.phase == PH_FEW) {
    const int cnt = (int)min(sp.few_count[row], (uint32_t)SMALL_MAX);
    for (int e = threadIdx.x; e < cnt; e += SNT) {
      sh.one.s_key[e] = sp.few_key[(size_t)row * SMALL_MAX + e];
      sh.one.s_id[e] = sp.few_id[(size_t)row * SMALL_MAX + e];
    }
    __syncthreads();
    const bool use_top_p = tp >= 0.0f && tp < 1.0f && S.n > 1u;
    sample_few(sh.one, cnt, use_top_p, tp, r, out + row);
    to_host();
    return;
  }
  // a row whose cut or draw the launches did not cover (the caller's word on its rows was wrong), or is not through
  sample_row_one_block(sh.one, logits + (size_t)row * sz.ldl, sz.V, temperature[row], top_k[row], tp, r, out + row);
  to_host();
}

// ---- Rows that all keep at most SMALL_MAX candidates (0 < top-k <= 1,024), in two launches ----
// The k largest of a row are among the k largest of its pieces: every block leaves its piece's (and up to FEW_SPARE more,
// so that a coarse threshold will do), one block a row selects the row's k from those exactly, sorts them and does the
// reference's sequential arithmetic.  A threshold is found by radix descent over the same 64-bit sort key, 11
// bits a pass, with the histogram in LDS.  What bounds it is latency: each launch is a handful of passes over values that
// are in L2 after the first, each with two or three barriers; the descents above make five launches of it, each of which
// begins with where the one before it left off.  8 rows of 128,256 logits, top-k 40, top-p 0.95: 9.5 + 14.9 us (the descents:
// 73 us in seven launches).  Of the 14.9 us, by clock readings inside the kernel: the pieces' results 2, their candidates 1.6,
// the selection 4.3, sorting and exponentials 2, the sums in order 3 (7 when every value went from lane to lane); start and
// end of the launch are not among them.
constexpr int FEW_SPARE = 128, FEW_STRIDE = SMALL_MAX + FEW_SPARE;
constexpr int FEW_BITS = 11, FEW_BINS = 1 << FEW_BITS;

struct FewSpace {
  float* piece_best;       // [row][pieces] ...
  int* piece_arg;
  uint32_t* piece_finite;
  uint32_t* piece_count;   // candidates left
  uint32_t* key;           // [row][pieces][FEW_STRIDE]
  int* id;
  size_t bytes;
};

int most_pieces(int R) {
  const int want = ceil_div(512, R);
  return want > MAX_PIECES ? MAX_PIECES : want;
}

FewSpace carve_few(void* base, int R) {
  FewSpace s;
  size_t at = 0;
  auto take = [&](size_t bytes) { char* q = (char*)((uintptr_t)base + at); at += round16(bytes); return q; };
  const size_t n = (size_t)R * most_pieces(R);
  s.piece_best = (float*)take(n * 4);
  s.piece_arg = (int*)take(n * 4);
  s.piece_finite = (uint32_t*)take(n * 4);
  s.piece_count = (uint32_t*)take(n * 4);
  s.key = (uint32_t*)take(n * FEW_STRIDE * 4);
  s.id = (int*)take(n * FEW_STRIDE * 4);
  s.bytes = at;
  return s;
}

struct alignas(8) FewShared {
  uint32_t hist[FEW_BINS];
  uint32_t wave_sum[PNT / WAVE];
  uint32_t bin, above, at_bin, count;
  float bv[PNT / WAVE];
  int bi[PNT / WAVE];
  uint32_t nv[PNT / WAVE];
};

// The largest threshold c (a sort key with zeros below some digit) at which at least k and at most `most` >= k of the
// values stand at or above it; `each(f)` calls f(sort key) for the values of the block's NT threads.  Fewer than k values:
// 0.  With most == k the answer is exact: sort keys are all different.  A caller that knows k values whose bits from `hi` (32 or
// more) on are `prefix`, and none above them, says so.  ALIKE: a wave's values are often of one bin (in order, or equal), where an
// add a lane takes its turn (90,000 of them some 90 us): the lanes of the first one's bin add as one.
template <int NT, bool ALIKE = false, typename Each>
__device__ __forceinline__ u64 few_threshold(FewShared& sh, uint32_t k, uint32_t most, int key_bits, Each&& each, u64 prefix = 0,
                                             int hi = 64) {
  constexpr int PER = FEW_BINS / NT;
  uint32_t above = 0;                                   // values above the prefix's range
  for (;;) {
    const int lo = hi - FEW_BITS;                       // (0 or more: an id has at most 22 bits, see apc_sample_rows)
    __syncthreads();
#pragma unroll
    for (int g = 0; g < PER; ++g) sh.hist[threadIdx.x + g * NT] = 0;
    if (threadIdx.x == 0) sh.bin = 0xffffffffu;
    __syncthreads();
    each([&](u64 c) {
      if (hi < 64 && (c >> hi) != (prefix >> hi)) return;
      const uint32_t bin = (uint32_t)(c >> lo) & (FEW_BINS - 1);
      uint32_t n = 1;
      if constexpr (ALIKE) {
        const uint32_t first = __builtin_amdgcn_readfirstlane(bin);
        const u64 same = __ballot(bin == first);
        if (bin == first) {
          if ((int)(threadIdx.x % WAVE) != __ffsll(same) - 1) return;
          n = (uint32_t)__popcll(same);
        }
      }
      atomicAdd(&sh.hist[bin], n);
    });
    __syncthreads();
    // threads in descending order of the bins
    const int top = FEW_BINS - 1 - PER * (int)threadIdx.x, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    uint32_t h[PER], own = 0;
#pragma unroll
    for (int g = 0; g < PER; ++g) own += h[g] = sh.hist[top - g];
    uint32_t v = own;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const uint32_t up = __shfl_up(v, o, WAVE);
      if (lane >= o) v += up;
    }
    if (lane == WAVE - 1) sh.wave_sum[wave] = v;
    __syncthreads();
    uint32_t before = above + v - own;
#pragma unroll
    for (int w = 0; w < NT / WAVE; ++w)
      if (w < wave) before += sh.wave_sum[w];
#pragma unroll
    for (int g = 0; g < PER; ++g) {
      if (before < k && k <= before + h[g]) sh.bin = top - g, sh.above = before, sh.at_bin = h[g];
      before += h[g];
    }
    __syncthreads();
    if (sh.bin == 0xffffffffu) return 0;                // (the first pass only: fewer than k values)
    prefix |= (u64)sh.bin << lo;
    above = sh.above;
    if (above + sh.at_bin <= most || lo <= 64 - key_bits) return prefix;
    hi = lo;
  }
}

__device__ __forceinline__ void first_max(float& best, int& best_i, float ov, int oi) {
  if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
}

template <typename Options>
__global__ __launch_bounds__(PNT) void sample_few_pieces_kernel(const float* __restrict__ logits, SampleShape sz, Options opt, FewSpace sp) {
  __shared__ FewShared sh;
  const int row = blockIdx.y, piece = blockIdx.x;
  const float* lg = logits + (size_t)row * sz.ldl;
  const float temperature = opt.temperature[row], t = fmaxf(temperature, 1e-5f);
  const int tk = opt.top_k[row];
  const int i0 = piece * sz.chunk, i1 = min(sz.V, i0 + sz.chunk);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t nfin = 0;
  for_piece(lg, sz.vec, i0, i1, [&](int i, float v) {
    if (v > best) { best = v; best_i = i; }
    nfin += finite_f(v) ? 1u : 0u;
  });
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    first_max(best, best_i, __shfl_xor(best, o, WAVE), __shfl_xor(best_i, o, WAVE));
    nfin += __shfl_xor(nfin, o, WAVE);
  }
  if (threadIdx.x % WAVE == 0) {
    sh.bv[threadIdx.x / WAVE] = best;
    sh.bi[threadIdx.x / WAVE] = best_i;
    sh.nv[threadIdx.x / WAVE] = nfin;
  }
  if (threadIdx.x == 0) sh.count = 0;
  __syncthreads();
  nfin = 0;
  for (int w = 0; w < PNT / WAVE; ++w) {
    first_max(best, best_i, sh.bv[w], sh.bi[w]);
    nfin += sh.nv[w];
  }
  const size_t at = (size_t)row * sz.pieces + piece;
  if (threadIdx.x == 0) {
    sp.piece_best[at] = best;
    sp.piece_arg[at] = best_i;
    sp.piece_finite[at] = nfin;
  }
  if (tk <= 0 || tk > SMALL_MAX || temperature <= 1e-5f) return;   // the last launch knows what to do with the row
  auto each = [&](auto f) {
    for_piece(lg, sz.vec, i0, i1, [&](int i, float x) {
      if (finite_f(x)) f(sort_key(key_of(x / t), i, sz.id_bits, 0));
    });
  };
  const u64 from = nfin <= (uint32_t)(tk + FEW_SPARE) ? 0 : few_threshold<PNT>(sh, tk, tk + FEW_SPARE, 32 + sz.id_bits, each);
  each([&](u64 c) {
    if (c < from) return;
    const uint32_t j = atomicAdd(&sh.count, 1u);        // (at most tk + FEW_SPARE of them)
    sp.key[at * FEW_STRIDE + j] = (uint32_t)(c >> 32);
    sp.id[at * FEW_STRIDE + j] = id_of_sort_key(c, sz.id_bits, 0);
  });
  __syncthreads();
  if (threadIdx.x == 0) sp.piece_count[at] = sh.count;
}

// run[i] = start + sign (a[0] + .. + a[i]) for the first n values, one after the other (the order of the reference's sums), by
// one wave.  All lanes add the same values, sixteen out of LDS at a time and the next sixteen asked for meanwhile; there is room
// behind n in both up to a multiple of 16.  (A value handed round from lane to lane costs 110 cycles, and code written out 64
// times more than the sums, since a block alone brings in every line of it.)
__device__ __forceinline__ void sums_in_order(const float* a, float* run, int n, float start, float sign) {
  const int lane = threadIdx.x % WAVE;
  const f32x4* a4 = reinterpret_cast<const f32x4*>(a);
  float acc = start;
  f32x4 next[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) next[q] = a4[q];
#pragma unroll 1
  for (int i = 0; i < n; i += 16) {
    f32x4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = next[q];
    const int then = min(i + 16, (n - 1) / 16 * 16) / 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) next[q] = a4[then + q];
    float mine = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      acc += sign * v[u / 4][u % 4];                     // (what stands behind n is added behind all that counts)
      mine = lane == u ? acc : mine;
    }
    if (lane < 16) run[i + lane] = mine;
  }
  __builtin_amdgcn_wave_barrier();
}

// The token among the cnt candidates in sh.s_key2 / sh.s_id2, in order: as `sample_few`, with the exponentials and quotients by
// all threads and the sums in order by one wave.  share, sums: room for cnt floats and up to a multiple of 16 behind them.
template <int NT, typename Leave>
__device__ __forceinline__ void draw_in_order(SampleShared& sh, float* share, float* sums, int cnt, bool use_top_p, float tp, float uniform,
                                              Leave&& leave) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  float* e = reinterpret_cast<float*>(sh.s_key);
  const float vmax = value_of(sh.s_key2[0]);
  for (int i = threadIdx.x; i < cnt; i += NT) e[i] = expf(value_of(sh.s_key2[i]) - vmax);
  __syncthreads();
  if (wave != 0) return;
  // The weights' sum, the shares' sum up to top-p, and the uniform number less the shares of the m that are left: three times
  // the same code (over values that differ), which a block fetches once.  The sum of the first m is one of the first pass's.
  float* run = reinterpret_cast<float*>(sh.s_id);
  int m = cnt, pick = 0;
  float sum = 0.f;
#pragma unroll 1
  for (int pass = 0; pass < 3; ++pass) {
    if (pass == 1) {
      if (!use_top_p) continue;
      if (sum == 0.f || !finite_f(sum)) {
        const int some = (int)ceilf(tp * (float)m);
        m = some < 1 ? 1 : (some > m ? m : some);
        sum = sums[m - 1];
        continue;
      }
    }
    for (int i = lane; i < m; i += WAVE) share[i] = pass == 0 ? e[i] : pass == 2 && sum == 0.f ? 1.0f / (float)m : e[i] / sum;
    __builtin_amdgcn_wave_barrier();
    float* to = pass == 0 ? sums : run;
    sums_in_order(share, to, m, pass == 2 ? uniform : 0.f, pass == 2 ? -1.f : 1.f);
    if (pass == 0) {
      sum = sums[m - 1];
      continue;
    }
    // the first candidate at which top-p is reached, or at which nothing is left
    int first = m - 1;
    for (int i0 = 0; i0 < m; i0 += WAVE) {
      const int i = i0 + lane;
      const unsigned long long hit = __ballot(i < m && (pass == 1 ? run[i] >= tp : run[i] <= 0.f));
      if (hit) {
        first = i0 + __ffsll(hit) - 1;
        break;
      }
    }
    if (pass == 1) m = first + 1, sum = sums[first];
    else pick = first;
  }
  if (lane == 0) leave(sh.s_id2[pick]);
}

constexpr int FEW_HELD = 6144;           // candidates of a row that are held in LDS (all of them up to top-k 64)
struct FewEnd {
  FewShared select;
  SampleShared one;
  u64 held[FEW_HELD];
  uint32_t from[MAX_PIECES + 1];         // where the candidates of a piece begin
  float sums[SMALL_MAX];                 // running sums of the weights
};

// `out_host` (may be null): host memory that the ids are written to as well.
template <typename Options>
__global__ __launch_bounds__(SNT) void sample_few_end_kernel(const float* __restrict__ logits, SampleShape sz, Options opt, FewSpace sp,
                                                             int* __restrict__ out, int* __restrict__ out_host) {
  __shared__ FewEnd sh;
  const int row = blockIdx.x, tk = opt.top_k[row];
  const float T = opt.temperature[row], tp = opt.top_p[row], uniform = opt.uniform[row];
  auto leave = [&](int id) {
    out[row] = id;
    if (out_host) out_host[row] = id;
  };
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t n = 0;
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  if (lane < sz.pieces) {                               // every wave for itself, a piece a lane
    const size_t at = (size_t)row * sz.pieces + lane;
    best = sp.piece_best[at];
    best_i = sp.piece_arg[at];
    n = sp.piece_finite[at];
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    first_max(best, best_i, __shfl_xor(best, o, WAVE), __shfl_xor(best_i, o, WAVE));
    n += __shfl_xor(n, o, WAVE);
  }
  if (n == 0u || T <= 1e-5f) {
    if (threadIdx.x == 0) leave(n == 0u || best_i == 0x7fffffff ? 0 : best_i);
    return;
  }
  const bool cut = tk > 0 && n > (uint32_t)tk;
  const uint32_t keep = cut ? (uint32_t)tk : n;
  const bool use_top_p = tp >= 0.0f && tp < 1.0f && keep > 1u;
  if (tk <= 0 || tk > SMALL_MAX || !(cut || use_top_p)) {
    // the caller's word on the row was wrong, or fewer candidates than top-k keeps and no top-p: drawn in id order
    sample_row_one_block(sh.one, logits + (size_t)row * sz.ldl, sz.V, T, tk, tp, uniform, out + row);
    __syncthreads();
    if (out_host && threadIdx.x == 0) out_host[row] = *(volatile int*)(out + row);
    return;
  }
  if (wave == 0) {
    uint32_t v = lane < sz.pieces ? sp.piece_count[(size_t)row * sz.pieces + lane] : 0u;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const uint32_t up = __shfl_up(v, o, WAVE);
      if (lane >= o) v += up;
    }
    if (lane == 0) sh.from[0] = 0;
    if (lane < MAX_PIECES) sh.from[lane + 1] = v;
  }
  __syncthreads();
  const uint32_t total = sh.from[MAX_PIECES];
  const bool held = total <= (uint32_t)FEW_HELD;
  auto candidate = [&](int p, int j) {
    const size_t at = ((size_t)row * sz.pieces + p) * FEW_STRIDE + j;
    return sort_key(sp.key[at], sp.id[at], sz.id_bits, 0);
  };
  if (held) {                                           // the first 128 of all of a wave's pieces are asked for together
    constexpr int MINE = MAX_PIECES / (SNT / WAVE);
    u64 c[MINE][2];
#pragma unroll
    for (int g = 0; g < MINE; ++g)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // (places that hold no candidate are read too: there is room for FEW_STRIDE in every piece)
        c[g][u] = candidate(min(wave + g * (SNT / WAVE), sz.pieces - 1), lane + u * WAVE);
      }
#pragma unroll
    for (int g = 0; g < MINE; ++g) {
      const int p = wave + g * (SNT / WAVE), count = (int)(sh.from[p + 1] - sh.from[p]);
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (lane + u * WAVE < count) sh.held[sh.from[p] + lane + u * WAVE] = c[g][u];
      for (int j = lane + 2 * WAVE; j < count; j += WAVE) sh.held[sh.from[p] + j] = candidate(p, j);
    }
    __syncthreads();
  }
  auto each = [&](auto f) {                             // every candidate of the row's pieces
    if (held) {
      for (int i = threadIdx.x; i < (int)total; i += SNT) f(sh.held[i]);
    } else {
      for (int p = wave; p < sz.pieces; p += SNT / WAVE)
        for (int j = lane; j < (int)(sh.from[p + 1] - sh.from[p]); j += WAVE) f(candidate(p, j));
    }
  };
  u64* picked = reinterpret_cast<u64*>(sh.select.hist);  // (the histogram is done with by then)
  static_assert(sizeof(sh.select.hist) >= SMALL_MAX * sizeof(u64), "the candidates that are kept fit the histogram's room");
  if (threadIdx.x == 0) sh.select.count = 0;
  const u64 from = cut ? few_threshold<SNT>(sh.select, keep, keep, 32 + sz.id_bits, each) : 0;
  __syncthreads();
  each([&](u64 c) {
    if (c < from) return;
    const uint32_t j = atomicAdd(&sh.select.count, 1u);
    if (j < (uint32_t)SMALL_MAX) picked[j] = c;
  });
  __syncthreads();
  const int cnt = (int)keep;
  for (int e = threadIdx.x; e < cnt; e += SNT) {
    const u64 mine = picked[e];
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < cnt; ++j) rank += picked[j] > mine ? 1 : 0;
    sh.one.s_key2[rank] = (uint32_t)(mine >> 32);
    sh.one.s_id2[rank] = id_of_sort_key(mine, sz.id_bits, 0);
  }
  __syncthreads();
  draw_in_order<SNT>(sh.one, reinterpret_cast<float*>(sh.select.hist), sh.sums, cnt, use_top_p, tp, uniform, leave);   // (picked has been sorted)
}

// ---- The same, with a bound that the largest values of groups give ----
// Of a row's groups of values, at least k have a largest value at or above the k-th largest of these; so the row's k largest
// stand at or above it too, and only in groups whose largest does.  The first launch reads the row once and leaves every
// wave's largest value; the second finds the bound among at most BOUND_SET of them (waves, or four waves together), reads again
// the few groups that reach it (for k of 40 some 45 of 512, of 256 values each) and puts what it finds in order by counting who
// stands above whom.  A row whose large values lie close together (all in one group, or all equal) has more than HEAD_HELD
// there: of all waves by their largest value (of equal ones the earlier pieces') only those that fewer than k others come in front
// of can hold one of the k largest, some k of them, and the radix descent over these stops at a few values more than k.
// What bounds it is latency: the first launch is one pass where the pair above makes three, the second has some 45 groups' values to
// look at instead of 1,300 to 5,000 candidates, and divides only those by the temperature that may stand at the bound.  Both launches,
// rows of 128,256 random logits, top-p 0.95, pair above / this one, us: 8 rows top-k 8 19.4 / 14.1, 40 25.2 / 16.2, 85 30.2 / 22.5; 64
// rows 38.6 / 17.6, 44.6 / 23.1, 54.0 / 33.2; from the call to the ids, 8 rows of top-k 40, 47.5 / 39.7 (without the divisions that are
// spared).  8 rows of equal values, top-k 40, 43.9 / 40.3 (476 with a descent over all of the row); where the large values are some
// thousand neighbours, which logits are not, the pair above stays ahead: in descending order 28.2 / 31.7, top-k 85 32.2 / 42.4.
// The host has to know the rows' top-k, and one of more than two thirds of the set keeps the pair above: 85 of 128 fours of waves (up to
// 16 rows of 128,256), 170 of 256 waves (17 to 32 rows of 65,536, 32 of 128,256).
constexpr int BOUND_SET = 256, HEAD_HELD = 512, HEAD_WAVES = PNT / WAVE;
struct HeadSpace {
  float* piece_best;       // [row][pieces] ...
  int* piece_arg;
  uint32_t* piece_finite;
  uint32_t* wave_key;      // [row][pieces][HEAD_WAVES] key of the largest finite value, 0: none
};
// (in carve_few's memory: the candidates' place holds the waves' keys)
HeadSpace head_space(const FewSpace& fs) { return HeadSpace{fs.piece_best, fs.piece_arg, fs.piece_finite, fs.key}; }

__global__ __launch_bounds__(PNT) void sample_head_pieces_kernel(const float* __restrict__ logits, SampleShape sz, HeadSpace sp) {
  __shared__ float bv[HEAD_WAVES];
  __shared__ int bi[HEAD_WAVES];
  __shared__ uint32_t nv[HEAD_WAVES];
  const int row = blockIdx.y, piece = blockIdx.x, wave = threadIdx.x / WAVE;
  const float* lg = logits + (size_t)row * sz.ldl;
  const int i0 = piece * sz.chunk, i1 = min(sz.V, i0 + sz.chunk);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t nfin = 0, top = 0;
  for_piece(lg, sz.vec, i0, i1, [&](int i, float v) {
    if (v > best) { best = v; best_i = i; }
    if (finite_f(v)) ++nfin, top = max(top, key_of(v));
  });
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    first_max(best, best_i, __shfl_xor(best, o, WAVE), __shfl_xor(best_i, o, WAVE));
    nfin += __shfl_xor(nfin, o, WAVE);
    top = max(top, (uint32_t)__shfl_xor((int)top, o, WAVE));
  }
  const size_t at = (size_t)row * sz.pieces + piece;
  if (threadIdx.x % WAVE == 0) {
    bv[wave] = best;
    bi[wave] = best_i;
    nv[wave] = nfin;
    sp.wave_key[at * HEAD_WAVES + wave] = top;
  }
  __syncthreads();
  if (threadIdx.x >= HEAD_WAVES) return;
  best = bv[threadIdx.x], best_i = bi[threadIdx.x], nfin = nv[threadIdx.x];
#pragma unroll
  for (int o = HEAD_WAVES / 2; o > 0; o >>= 1) {
    first_max(best, best_i, __shfl_xor(best, o, HEAD_WAVES), __shfl_xor(best_i, o, HEAD_WAVES));
    nfin += __shfl_xor(nfin, o, HEAD_WAVES);
  }
  if (threadIdx.x == 0) {
    sp.piece_best[at] = best;
    sp.piece_arg[at] = best_i;
    sp.piece_finite[at] = nfin;
  }
}

// Whether the two kernels above and below take rows cut like this that keep up to `most` candidates: half as many groups again to
// bound them with (fewer leave a bound that many values reach).
__host__ __device__ int bound_set(const SampleShape& sz) {
  const int waves = sz.pieces * HEAD_WAVES;
  return waves <= BOUND_SET ? waves : waves / 4;
}
bool head_takes(const SampleShape& sz, int most) { return most * 3 <= bound_set(sz) * 2; }

// A value below this one, divided by t, has a key below `key` (rounded either way; spares the division for most values).
__device__ __forceinline__ float floor_of(uint32_t key, float t) {
  constexpr float MOST = 3.402823466e+38f;
  if (key < key_of(-MOST)) return -INFINITY;
  const float v = fminf(fminf(value_of(key), MOST) * t, MOST);
  return v - fabsf(v) * 1e-6f - 1e-37f;
}

struct HeadEnd {
  FewShared select;
  SampleShared one;
  uint32_t bound[BOUND_SET];
  u64 held[HEAD_HELD];
  int group[MAX_PIECES * HEAD_WAVES];
  int groups;
  uint32_t least, most;
  float sums[HEAD_HELD];                 // running sums of the weights
};

__global__ __launch_bounds__(PNT) void sample_head_end_kernel(const float* __restrict__ logits, SampleShape sz, RowValues opt, HeadSpace sp,
                                                              int* __restrict__ out, int* __restrict__ out_host) {
  __shared__ HeadEnd sh;
  const int row = blockIdx.x, tk = opt.top_k[row];
  const float T = opt.temperature[row], t = fmaxf(T, 1e-5f), tp = opt.top_p[row], uniform = opt.uniform[row];
  const float* lg = logits + (size_t)row * sz.ldl;
  auto leave = [&](int id) {
    out[row] = id;
    if (out_host) out_host[row] = id;
  };
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int waves = sz.pieces * HEAD_WAVES;
  const uint32_t* wave_key = sp.wave_key + (size_t)row * waves;
  auto scaled = [&](uint32_t key) { return key ? key_of(value_of(key) / t) : 0u; };
  static_assert(MAX_PIECES * HEAD_WAVES <= PNT, "a thread looks at one wave's key");
  const uint32_t mine = (int)threadIdx.x < waves ? wave_key[threadIdx.x] : 0u;
  const bool fours = waves > BOUND_SET;
  uint32_t own = 0;                                     // this thread's of the set
  if (!fours) own = mine;
  else if ((int)threadIdx.x < waves / 4) {
    const uint4 q = reinterpret_cast<const uint4*>(wave_key)[threadIdx.x];
    own = max(max(q.x, q.y), max(q.z, q.w));
  }
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  uint32_t n = 0;
  if (lane < sz.pieces) {                               // every wave for itself, a piece a lane
    const size_t at = (size_t)row * sz.pieces + lane;
    best = sp.piece_best[at];
    best_i = sp.piece_arg[at];
    n = sp.piece_finite[at];
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    first_max(best, best_i, __shfl_xor(best, o, WAVE), __shfl_xor(best_i, o, WAVE));
    n += __shfl_xor(n, o, WAVE);
  }
  if (n == 0u || T <= 1e-5f) {
    if (threadIdx.x == 0) leave(n == 0u || best_i == 0x7fffffff ? 0 : best_i);
    return;
  }
  const bool cut = tk > 0 && n > (uint32_t)tk;
  const uint32_t keep = cut ? (uint32_t)tk : n;
  const bool use_top_p = tp >= 0.0f && tp < 1.0f && keep > 1u;
  const int set = bound_set(sz);
  if (tk <= 0 || tk * 3 > set * 2 || !(cut || use_top_p)) {
    // the caller's word on the row was wrong, or fewer candidates than top-k keeps and no top-p: drawn in id order
    if (threadIdx.x >= SNT) return;                     // (whole waves: a barrier does not wait for those that have ended)
    sample_row_one_block(sh.one, lg, sz.V, T, tk, tp, uniform, out + row);
    __syncthreads();
    if (out_host && threadIdx.x == 0) out_host[row] = *(volatile int*)(out + row);
    return;
  }
  // the bound: the keep-th largest of the set.  The lowest byte says who is who, so no two are alike, and is then left out
  const uint32_t tag = BOUND_SET - 1 - threadIdx.x, who = (scaled(own) & ~(uint32_t)(BOUND_SET - 1)) | tag;
  if ((int)threadIdx.x < BOUND_SET) sh.bound[threadIdx.x] = (int)threadIdx.x < set ? who : 0u;
  if (threadIdx.x == 0) sh.groups = 0, sh.least = 0u, sh.select.count = 0;
  __syncthreads();
  if (cut) {
    if ((int)threadIdx.x < set) {
      int above = 0;
      const uint4* others = reinterpret_cast<const uint4*>(sh.bound);
#pragma unroll 8
      for (int q = 0; q < (set + 3) / 4; ++q) {
        const uint4 o = others[q];
        above += (o.x > who) + (o.y > who) + (o.z > who) + (o.w > who);
      }
      if (above == (int)keep - 1) sh.least = who & ~(uint32_t)(BOUND_SET - 1);
    }
    __syncthreads();
  }
  const uint32_t least = max(sh.least, 1u);
  const int listed = scaled(mine) >= least ? atomicAdd(&sh.groups, 1) : -1;
  if (listed >= 0) sh.group[listed] = threadIdx.x;
  __syncthreads();
  // f(sort key) for the finite values of these groups that may stand at the bound: a wave takes four rounds of a group at a time
  const int per = sz.vec ? 4 * PNT : PNT, rounds = ceil_div(sz.chunk, per);
  int items = sh.groups * rounds;
  float floor = floor_of(least, t);
  auto each = [&](auto f) {
    for (int q = wave * 4; q < items; q += PNT / WAVE * 4) {
      if (*(volatile uint32_t*)&sh.select.count > (uint32_t)HEAD_HELD) break;   // (more than there is room for: see below)
      float x[4][4];
      int at[4], end[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int item = min(q + u, items - 1), g = sh.group[item / rounds], piece = g / HEAD_WAVES, i0 = piece * sz.chunk;
        end[u] = q + u < items ? min(sz.V, i0 + sz.chunk) : 0;
        at[u] = i0 + item % rounds * per + (g % HEAD_WAVES * WAVE + lane) * (sz.vec ? 4 : 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][e] = INFINITY;
        if (sz.vec) {
          if (at[u] + 3 < end[u]) {
            const float4 v = *reinterpret_cast<const float4*>(lg + at[u]);
            x[u][0] = v.x, x[u][1] = v.y, x[u][2] = v.z, x[u][3] = v.w;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (at[u] + e < end[u]) x[u][e] = lg[at[u] + e];
          }
        } else if (at[u] < end[u]) {
          x[u][0] = lg[at[u]];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (x[u][e] >= floor && finite_f(x[u][e])) f(sort_key(key_of(x[u][e] / t), at[u] + e, sz.id_bits, 0));
    }
  };
  auto gather = [&](u64 from) {
    each([&](u64 c) {
      if (c < from) return;
      const uint32_t j = atomicAdd(&sh.select.count, 1u);
      if (j < (uint32_t)HEAD_HELD) sh.held[j] = c;
    });
    __syncthreads();
  };
  gather((u64)least << 32);
  if (sh.select.count > (uint32_t)HEAD_HELD) {          // (the same for all threads)
    // The waves that fewer than `keep` others come in front of; another one's values stand behind `keep` others.
    u64* order = reinterpret_cast<u64*>(sh.select.hist);
    static_assert(MAX_PIECES * HEAD_WAVES * sizeof(u64) <= sizeof(sh.select.hist), "room for all waves");
    const u64 me = (u64)scaled(mine) << 32 | (MAX_PIECES - threadIdx.x / HEAD_WAVES);
    const int n_listed = sh.groups;
    if (listed >= 0) order[listed] = me;
    __syncthreads();
    if (threadIdx.x == 0) sh.groups = 0, sh.select.count = 0, sh.least = 0xffffffffu, sh.most = 0;
    uint32_t front = 0;
    if (listed >= 0) {
#pragma unroll 8
      for (int q = 0; q < n_listed; ++q) front += order[q] > me;
    }
    __syncthreads();
    if (listed >= 0 && front < keep) {
      sh.group[atomicAdd(&sh.groups, 1)] = threadIdx.x;
      atomicMin(&sh.least, (uint32_t)(me >> 32));
      atomicMax(&sh.most, (uint32_t)(me >> 32));
    }
    __syncthreads();
    items = sh.groups * rounds;
    // Where there are `keep` such waves, `keep` values stand between the least and the largest of their keys: the bits that these two
    // have in common need no pass.
    const uint32_t low = sh.groups >= (int)keep ? sh.least : 1u;
    const int hi = low == sh.most ? 32 : 64 - __clz((int)(low ^ sh.most));
    const u64 prefix = hi < 64 ? (u64)sh.most << 32 >> hi << hi : 0;
    floor = floor_of(low, t);
    const u64 from = few_threshold<PNT, true>(sh.select, keep, keep + FEW_SPARE, 32 + sz.id_bits, each, prefix, hi);
    floor = floor_of((uint32_t)(from >> 32), t);
    gather(from);
  }
  const int found = (int)sh.select.count;
  for (int e = threadIdx.x; e < found; e += PNT) {
    const u64 c = sh.held[e];
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < found; ++j) rank += sh.held[j] > c ? 1 : 0;
    if (rank < (int)keep) {
      sh.one.s_key2[rank] = (uint32_t)(c >> 32);
      sh.one.s_id2[rank] = id_of_sort_key(c, sz.id_bits, 0);
    }
  }
  __syncthreads();
  draw_in_order<PNT>(sh.one, reinterpret_cast<float*>(sh.select.hist), sh.sums, (int)keep, use_top_p, tp, uniform, leave);
}

std::mutex pass_attr_lock;
bool pass_attr_set[64];

SampleShape shape_of(const float* logits, int ldl, int n_rows, int V) {
  SampleShape sz;
  sz.ldl = ldl;
  sz.V = V;
  sz.R = n_rows;
  cut_row(n_rows, V, &sz.pieces, &sz.chunk);
  sz.vec = ((uintptr_t)logits % 16 == 0 && ldl % 4 == 0) ? 1 : 0;
  sz.id_bits = 1;
  while (sz.id_bits < 31 && (1u << sz.id_bits) < (unsigned)V) ++sz.id_bits;
  sz.key_digits = ceil_div(32 + sz.id_bits, DIGIT_BITS);
  sz.id_digits = ceil_div(sz.id_bits, DIGIT_BITS);
  return sz;
}

template <typename Options>
int launch_few(const float* logits, const SampleShape& sz, const Options& opt, void* scratch, int* out, int* out_host, hipStream_t stream) {
  const FewSpace fs = carve_few(scratch, sz.R);
  hipLaunchKernelGGL(sample_few_pieces_kernel<Options>, dim3(sz.pieces, sz.R), dim3(PNT), 0, stream, logits, sz, opt, fs);
  APC_LAUNCH_CHECK();
  hipLaunchKernelGGL(sample_few_end_kernel<Options>, dim3(sz.R), dim3(SNT), 0, stream, logits, sz, opt, fs, out, out_host);
  APC_LAUNCH_CHECK();
  return 0;
}

int launch_head(const float* logits, const SampleShape& sz, const RowValues& opt, void* scratch, int* out, int* out_host, hipStream_t stream) {
  const HeadSpace sp = head_space(carve_few(scratch, sz.R));
  hipLaunchKernelGGL(sample_head_pieces_kernel, dim3(sz.pieces, sz.R), dim3(PNT), 0, stream, logits, sz, sp);
  APC_LAUNCH_CHECK();
  hipLaunchKernelGGL(sample_head_end_kernel, dim3(sz.R), dim3(PNT), 0, stream, logits, sz, opt, sp, out, out_host);
  APC_LAUNCH_CHECK();
  return 0;
}

int allow_pass_lds(int dev) {
  std::lock_guard<std::mutex> hold(pass_attr_lock);
  if (!pass_attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)sample_pass_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)sizeof(PassShared));
    if (e != hipSuccess) return (int)e;
    pass_attr_set[dev] = true;
  }
  return 0;
}

// `values`: the options, if they are on the host (then `opt` is not looked at)
int launch_descents(const float* logits, const SampleShape& sz, RowOptions opt, const RowValues* values, void* scratch, int* out,
                    int* out_host, int cuts, hipStream_t stream) {
  const SampleSpace sp = carve(scratch, sz.R);
  const dim3 grid(sz.pieces, sz.R);
  if (values) {
    opt = RowOptions{sp.options->temperature, sp.options->top_p, sp.options->uniform, sp.options->top_k};
    hipLaunchKernelGGL(sample_max_kernel<RowValues>, grid, dim3(PNT), 0, stream, logits, sz, *values, sp);
  } else {
    hipLaunchKernelGGL(sample_max_kernel<NoValues>, grid, dim3(PNT), 0, stream, logits, sz, NoValues{}, sp);
  }
  APC_LAUNCH_CHECK();
  int q = 0, prev_stage = -1, prev_digit = -1;
  for (int stage = 0; stage < N_SELECTS; ++stage) {
    int digits = sz.key_digits;
    if (stage == ST_TOPK && !(cuts & 1)) continue;
    if (stage == ST_TOPP && !(cuts & 2)) continue;
    if (stage == ST_DRAW) digits = (cuts & 3) ? sz.key_digits : sz.id_digits;
    for (int digit = 0; digit < digits; ++digit) {
      hipLaunchKernelGGL(sample_pass_kernel, grid, dim3(PNT), sizeof(PassShared), stream, logits, sz, opt.temperature,
                         opt.top_k, opt.top_p, opt.uniform, sp, q, stage, digit, prev_stage, prev_digit);
      APC_LAUNCH_CHECK();
      ++q;
      prev_stage = stage;
      prev_digit = digit;
    }
  }
  hipLaunchKernelGGL(sample_end_kernel, dim3(sz.R), dim3(SNT), 0, stream, logits, sz, opt.temperature, opt.top_k, opt.top_p,
                     opt.uniform, sp, q, prev_stage, prev_digit, out, out_host);
  APC_LAUNCH_CHECK();
  return 0;
}

uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  uint64_t z = x;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

}  // namespace

// KiB of working memory that apc_sample_rows wants for n_rows rows (it takes the one-block way without)
APC_EXPORT int apc_sample_rows_scratch_kib(int n_rows) {
  if (n_rows <= 0 || n_rows > 65535) return 0;
  const size_t bytes = carve(nullptr, n_rows).bytes, few = carve_few(nullptr, n_rows).bytes;
  return (int)(((bytes > few ? bytes : few) + 1023) / 1024);
}

// `cuts`: bit 0 set if some row may have top-k > 0, bit 1 if some row may have 0 <= top-p < 1, bit 2 if every row that
// samples has 0 < top-k <= 1,024.  Bits 0 and 2 together take the two launches of sample_few_pieces_kernel and
// sample_few_end_kernel, with or without top-p, and the working memory in carve_few's layout; everything else the
// descents, in carve's.  A caller that does not know its rows passes 3.  A row for which the caller's word is wrong
// still gets its token, the slow way.
APC_EXPORT int apc_sample_rows(const float* logits, int ldl, int n_rows, int V, const float* temperature,
                               const int* top_k, const float* top_p, const float* uniform, int* out, void* scratch,
                               size_t scratch_bytes, int cuts, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (V <= 0 || ldl < V) return APC_ERR_BAD_ARG;
  int dev = -1;
  if (scratch) {
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
  }
  // (a row's weights add up in 64 bits: 2^40 a candidate at most, so 2^22 candidates stay far inside)
  if (!scratch || n_rows > 65535 || dev < 0 || dev >= 64 || V > (1 << 22)) {
    hipLaunchKernelGGL(sample_rows_kernel, dim3(n_rows), dim3(SNT), 0, stream, logits, ldl, V, temperature, top_k,
                       top_p, uniform, out);
    APC_LAUNCH_CHECK();
    return 0;
  }
  const bool few = (cuts & 5) == 5;
  if (((uintptr_t)scratch & 15u) || scratch_bytes < (few ? carve_few(nullptr, n_rows).bytes : carve(nullptr, n_rows).bytes))
    return APC_ERR_BAD_ARG;
  if (!few)
    if (const int rc = allow_pass_lds(dev)) return rc;
  const SampleShape sz = shape_of(logits, ldl, n_rows, V);
  if (few) return launch_few(logits, sz, RowOptions{temperature, top_p, uniform, top_k}, scratch, out, nullptr, stream);
  return launch_descents(logits, sz, RowOptions{temperature, top_p, uniform, top_k}, nullptr, scratch, out, nullptr, cuts, stream);
}

// 1 if the entry point below bounds the rows' values by the largest ones of groups (sample_head_end_kernel) where no row that samples
// has a larger top-k than `most`, all of them between 1 and 1,024.
APC_EXPORT int apc_sample_rows_bounded(int n_rows, int V, int most) {
  return n_rows > 0 && n_rows <= BY_VALUE && V > 0 && V <= (1 << 22) && most > 0 && head_takes(shape_of(nullptr, V, n_rows, V), most) ? 1 : 0;
}

// The same for up to 64 rows with their options on the host: they go with the first launch, and the ids also to `out_host` (host
// memory that the device can write, or null), so that nothing is copied either way.  `options`: n_rows temperatures (float),
// top-p (float), top-k (int), seeds (uint64) and numbers of the generated token (int64), one behind the other; the uniform number
// of a row is that of (seed, number).  From the call to the ids on the host, 8 rows of 128,256: top-k 40 and top-p 0.95 85 -> 48
// us (of which the sums in order, 7 -> 3, are 4), top-p alone 142 -> 108.
APC_EXPORT int apc_sample_rows_host(const float* logits, int ldl, int n_rows, int V, const void* options, int* out, int* out_host,
                                    void* scratch, size_t scratch_bytes, int cuts, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  const bool few = (cuts & 5) == 5;
  if (V <= 0 || ldl < V || n_rows > BY_VALUE || !options || !scratch || ((uintptr_t)scratch & 15u) ||
      scratch_bytes < (few ? carve_few(nullptr, n_rows).bytes : carve(nullptr, n_rows).bytes))
    return APC_ERR_BAD_ARG;
  int dev = -1;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (V > (1 << 22) || dev < 0 || dev >= 64) return APC_ERR_UNSUPPORTED;
  RowValues opt = {};
  const size_t n = n_rows;
  const char* from = (const char*)options;
  memcpy(opt.temperature, from, 4 * n);
  memcpy(opt.top_p, from + 4 * n, 4 * n);
  memcpy(opt.top_k, from + 8 * n, 4 * n);
  for (size_t r = 0; r < n; ++r) {
    uint64_t seed, number;
    memcpy(&seed, from + 12 * n + 8 * r, 8);
    memcpy(&number, from + 20 * n + 8 * r, 8);
    opt.uniform[r] = (float)(splitmix64(splitmix64(seed) ^ ((number + 1) * 0xD6E8FEB86659FD93ull)) >> 40) / (float)(1 << 24);
  }
  const SampleShape sz = shape_of(logits, ldl, n_rows, V);
  if (few) {
    int most = 0;                                        // (greedy rows may ask for any)
    for (int r = 0; r < n_rows; ++r)
      if (opt.temperature[r] > 1e-5f) most = std::max(most, opt.top_k[r]);
    return most > 0 && head_takes(sz, most) ? launch_head(logits, sz, opt, scratch, out, out_host, stream)
                                            : launch_few(logits, sz, opt, scratch, out, out_host, stream);
  }
  if (const int rc = allow_pass_lds(dev)) return rc;
  return launch_descents(logits, sz, RowOptions{}, &opt, scratch, out, out_host, cuts, stream);
}
