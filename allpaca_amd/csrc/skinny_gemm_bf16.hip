// Matrix product for few rows (decode):  C[M,N] = A[M,K] . W[N,K]^T,  M <= 16, bfloat16 in, float32 sums.
//
// The step is bound by reading W once from HBM, so the kernel is a stream over W, which is stored in
// tiles of 16 rows x 32 columns laid out as the 64 lanes of a wave hold an operand of
// v_mfma_f32_16x16x32_bf16 (1 KiB a tile, tiles of a 16-row band in K order, bands in N order; rows and
// columns beyond N, K are zero):
//  * a block owns NB bands (16 NB output columns) and all of K; each of its WPB waves takes a contiguous
//    range of K and reads it in steps of 4 tiles per band: every load of W is 1 KiB of consecutive bytes and a
//    wave walks forward through one region of memory;
//  * the activations are the other operand, D[n][m], loaded once per step for all NB bands, so a lane ends with 4
//    consecutive n of one row m (SwiGLU: steps of 2 tiles).  One load takes 8 rows x 64 columns, whole lines of 128 bytes,
//    for a pair of tiles: lanes 0-7 of 16 hold the rows' part of the first tile, lanes 8-15 of the second.  Both tiles
//    are multiplied with it; the first one's sums count in columns 0-7 of the result, the second one's in 8-15, and
//    they are added at the end (9-16 rows: two groups of 8, the same sums).  Operands of 16 rows x 32 columns, as the
//    instruction takes them, are half lines, which come out of L2 at a third of the rate, and with up to 8 rows half of
//    them repeat a row: a step of one row at 1B shapes 743 -> 727 us, of 8 rows at 8B shapes 3.39 -> 3.32 ms;
//  * the loads of the next step are in flight while the current one is multiplied (two register sets that
//    swap roles; no branch around a load in the steady state);
//  * the waves' partial sums are added in wave order through LDS, then the epilogue runs: store (bfloat16 or
//    float32), add into a float32 residual, SwiGLU of a gate band and an up band, or rotation of q and k and the
//    write of k and v into the paged cache (SK_QKV_ROPE, see SkRope).
//  * the RMS norm between a product that adds into the residual x and the product that reads the normalised row
//    is folded into the two (EMIT and PRE): the first writes, beside x, the row bfloat16(x[m,n] * g[n]) (g: the
//    norm's weight) and, per band of 16 columns, the sum of x^2 of each row; the second multiplies with that row
//    as it is and scales its sums by 1 / sqrt(mean(x^2) + eps), which it gets by adding the bands' sums in band
//    order.  That is the product of the normalised row up to where the rounding to bfloat16 falls, without a
//    kernel of its own for the norm.
// The order of additions for an output depends on N and K, never on which other rows are in the batch: a
// decoded row is the same alone and in any batch of up to 16 rows.
// Reference counterpart: gemv_nt_bf16_{wide,wide_rows,splitk}_kernel, hip/src/kernels.cpp:3555-3700
// (no matrix cores, row-major weights); the product is matmul_nt, crates/allpaca-cpu/src/kernels.rs:97-128.
#include "mfma.h"

constexpr int SK_U = 4;              // tiles (32 k each) per band per step
constexpr int TILE_ELEMS = 16 * 32;  // elements of a tile

enum { SK_STORE_BF16 = 0, SK_STORE_F32 = 1, SK_ACC_F32 = 2, SK_SWIGLU = 3, SK_QKV_ROPE = 4, SK_ACT = 5 };

template <int MG, int NB, int U>
struct SkRegs {
  Frag w[NB][U];
  Frag a[MG][U / 2];
};

// what lane l ^ 8 holds
__device__ __forceinline__ floatx4 eight_lanes_on(const floatx4& v) {
  floatx4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float x = v[r];  // (a bit cast of the element itself takes element 0)
    o[r] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x128, 0xf, 0xf, true));  // row_ror:8
  }
  return o;
}

// NB: weight bands per block (for SwiGLU: 2 = one gate band and the up band of the same outputs)
// What the folded norm needs.  ss: sums of x^2 per row and band, [16 rows][ld_ss] floats, ld_ss = n_ss rounded up
// to a multiple of 4.  PRE (this product reads a row that an EMIT product left): ss, n_ss, eps.  EMIT (SK_ACC_F32
// only): g = the next norm's weight [N], raw = where the row bfloat16(x * g) goes [M, ld_raw], ss = where this
// product's n_ss = ceil(N / 16) bands leave their sums.
constexpr int SS_LOADS = 8;  // 16-byte loads of sums a lane may have to make (PRE): n_ss <= 4 * 4 * WPB * SS_LOADS
struct SkNorm {
  float* ss;
  int n_ss;
  int ld_ss;
  float eps;
  const float* g;
  bf16_t* raw;
  int ld_raw;
  int act = 0;   // SK_ACT: the activation on the sums (see activation_f), bfloat16 out
};

// SK_QKV_ROPE: the product that gives q, k and v of a row also turns q and k by the row's position and writes k
// and v into the paged cache, so no kernel of its own does that.  W is [(H + 2 Hk) d, K], heads in the order q, k, v;
// the whole head is rotated (pairs (e, e + d/2)); d is a multiple of 32.  A block takes the bands j and j + d/32 of
// one head, so a lane of the finishing wave holds both elements of 4 pairs.  Rotated q goes to C; k to
// cache[page][0][kv head][slot][:], v to cache[page][1][kv head][:][slot], page = block_table[row_seg][pos / P],
// slot = pos % P.  The sums are rounded to bfloat16 before the rotation, as a product that stores them would.
struct SkRope {
  const float* cos_sin;    // [positions][2][d / 2]
  const int* positions;    // [M]
  const int* row_seg;      // [M]
  const int* block_table;  // [segments][max_blocks]
  int max_blocks;
  bf16_t* cache;
  int P, H, Hk, d;
};

// Tiles per band and step, and the waves a SIMD that the compiler is asked to leave registers for (512 a lane in all).
// SwiGLU on a wide layer has more blocks than compute units and each block streams 2 bands: with steps of 2 tiles a wave
// needs no more than 128 registers, two blocks of 8 waves share a unit, and one block's first loads and final reduction
// hide behind the other's stream (8B shapes, 8 rows: 48.0 -> 44.4 us; the bytes in flight per unit stay the same).  For 9-16
// rows this has to be asked for: left to itself the compiler took 134 registers with a folded norm, one block a unit (with
// it, and the norm's sums added behind the stream, 9 rows at 8B shapes 42.2 -> 38.9 us, 16 rows 44.3 -> 40.9; q, k and v of
// 16 rows stored 18.0 -> 16.4).
constexpr int sk_step(int mode) { return mode == SK_SWIGLU ? 2 : SK_U; }
constexpr int sk_waves(int mg, int mode, int nb, int wpb, bool pre) {
  if (mode == SK_SWIGLU || nb == 1) return pre || mg == 2 ? 4 : mode == SK_ACC_F32 ? 5 : 6;
  return mg == 2 && wpb == 4 && !(mode == SK_QKV_ROPE && pre) ? 3 : 1;
}

template <int MG, int MODE, int NB, int WPB, bool PRE, bool EMIT>
__global__ __launch_bounds__(WPB * 64, sk_waves(MG, MODE, NB, WPB, PRE)) void skinny_gemm_kernel(const bf16_t* __restrict__ A, int lda,
                                                               const bf16_t* __restrict__ W,
                                                               const bf16_t* __restrict__ W2, int chunks,
                                                               void* __restrict__ C, int ldc, int M, int N, int K,
                                                               SkNorm norm, int vec_c, SkRope rope) {
  static_assert(MODE != SK_QKV_ROPE || NB == 2, "the two bands of a block hold the two halves of the pairs");
  static_assert(!EMIT || MODE == SK_ACC_F32, "only a product that adds into the residual emits the next norm's row");
  static_assert(!PRE || MODE != SK_ACC_F32, "a product that reads a normalised row stores its result");
  constexpr int U = sk_step(MODE);
  static_assert(MG == 1 || MG == 2, "one or two groups of 8 rows");
  static_assert(U % 2 == 0, "activations come two tiles at a time");
  __shared__ float red[WPB * NB * 256];
  __shared__ float row_ss[WPB * 16];
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int i = lane % 16, c = lane / 16;
  constexpr int OUT_BANDS = (MODE == SK_SWIGLU || MODE == SK_QKV_ROPE) ? 1 : NB;
  const int band0 = blockIdx.x * OUT_BANDS;
  const int bands = (N + 15) / 16;
  // SK_QKV_ROPE: head and first element of this lane's 4 pairs; position and segment of the finishing wave's row
  // are asked for before the stream starts, what depends on them behind its first loads
  int qkv_head = 0, qkv_e = 0, qkv_pos = 0, qkv_seg = 0;
  if constexpr (MODE == SK_QKV_ROPE) {
    const int hb = rope.d / 32;
    qkv_head = blockIdx.x / hb;
    qkv_e = (blockIdx.x % hb) * 16 + c * 4;
    if (wave == 0 && i < M) {
      qkv_pos = rope.positions[i];
      qkv_seg = rope.row_seg[i];
    }
  }

  // band pointers (bands beyond the matrix are clamped to the last: what they compute is never stored)
  const bf16_t* wb[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (MODE == SK_SWIGLU) wb[b] = (b == 0 ? W : W2) + (size_t)band0 * chunks * TILE_ELEMS + lane * 8;
    else if (MODE == SK_QKV_ROPE)
      wb[b] = W + (size_t)(qkv_head * (rope.d / 16) + blockIdx.x % (rope.d / 32) + b * (rope.d / 32)) * chunks * TILE_ELEMS + lane * 8;
    else wb[b] = W + (size_t)min(band0 + b, bands - 1) * chunks * TILE_ELEMS + lane * 8;
  }
  // row group g: lanes i < 8 take row g * 8 + i of a pair's first tile, lanes i >= 8 row g * 8 + i - 8 of its second
  // (in pieces of 8 elements: 15 rows of any stride an int holds fit 32 bits)
  uint32_t arow[MG];
#pragma unroll
  for (int g = 0; g < MG; ++g) arow[g] = (uint32_t)min(g * 8 + i % 8, M - 1) * (uint32_t)(lda / 8) + (i / 8) * 4 + c;

  // acc[b][g][t]: the tiles t of the pairs; of its 16 columns the group's rows are those of the lanes i / 8 == t
  floatx4 acc[NB][MG][2];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int g = 0; g < MG; ++g) acc[b][g][0] = acc[b][g][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto load_step = [&](SkRegs<MG, NB, U>& r, int ch) {  // tiles ch .. ch + U - 1, all inside K
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int b = 0; b < NB; ++b) r.w[b][u] = load_frag_once(wb[b] + (size_t)(ch + u) * TILE_ELEMS);
      if (u % 2 == 0) {
#pragma unroll
        for (int g = 0; g < MG; ++g) r.a[g][u / 2] = load_frag(A + (ch + u) * 32 + (size_t)arow[g] * 8);
      }
    }
  };
  auto compute = [&](const SkRegs<MG, NB, U>& r) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int g = 0; g < MG; ++g)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b][g][u % 2] = mfma16(r.w[b][u], r.a[g][u / 2], acc[b][g][u % 2]);
  };

  // this wave's range of tiles along K: [c_lo, c_hi); steps of 4 whole tiles, then single tiles
  const int full_chunks = K / 32;                       // tiles that lie wholly inside K (for the activations)
  const int per_wave = ((chunks + WPB - 1) / WPB + U - 1) / U * U;
  const int c_lo = min(wave * per_wave, chunks), c_hi = min(c_lo + per_wave, chunks);
  const int c_full_hi = min(c_hi, full_chunks);
  const int nsteps = c_full_hi > c_lo ? (c_full_hi - c_lo) / U : 0;
  // Steps are loaded two ahead (register sets r0, r1 take turns); no branch lies around a load in the steady loop,
  // so the waits for one set never wait for the other.
  SkRegs<MG, NB, U> r0, r1;
  if (nsteps > 0) load_step(r0, c_lo);
  if (nsteps > 1) load_step(r1, c_lo + U);
  // Behind the first loads of the stream, and needed only at the end: the sums of x^2 that the emitting product
  // left (PRE; the 4 * WPB (wave, c) pairs of the block take groups of 4 bands in turn, the pieces meet in LDS with
  // the partial sums of the product), and what the finishing wave of an output band adds to (residual, EMIT: g).
  // Two row groups' steps leave registers for two of these loads, which wait for their sum until the stream is through.
  float ss_piece = 0.f;
  floatx4 ss_v[2];
  const int ss_groups = PRE ? norm.ld_ss / 4 : 0;
  auto ss_load = [&](int j) {
    const int q = wave * 4 + c + j * WPB * 4;
    return q < ss_groups ? *reinterpret_cast<const floatx4*>(norm.ss + (size_t)i * norm.ld_ss + q * 4)
                         : floatx4{0.f, 0.f, 0.f, 0.f};
  };
  auto ss_add = [&](const floatx4& v, int j) {
    const int q = wave * 4 + c + j * WPB * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (q * 4 + e < norm.n_ss) ss_piece += v[e];
  };
  if constexpr (PRE && MG == 1) {
    floatx4 v[SS_LOADS];
#pragma unroll
    for (int j = 0; j < SS_LOADS; ++j) v[j] = ss_load(j);
#pragma unroll
    for (int j = 0; j < SS_LOADS; ++j) ss_add(v[j], j);
  } else if constexpr (PRE) {
    ss_v[0] = ss_load(0), ss_v[1] = ss_load(1);
  }
  constexpr int ITEMS = OUT_BANDS;  // bands to finish: wave w finishes band w
  const int fin_n = (band0 + wave) * 16 + c * 4;  // first of this lane's 4 columns if this wave finishes a band
  const bool fin_vec = vec_c && wave < ITEMS && i < M && fin_n + 3 < N;
  floatx4 c_old = floatx4{0.f, 0.f, 0.f, 0.f}, g_next = floatx4{0.f, 0.f, 0.f, 0.f};
  if (MODE == SK_ACC_F32 && fin_vec) {
    c_old = *reinterpret_cast<const floatx4*>((const float*)C + (size_t)i * ldc + fin_n);
    if constexpr (EMIT) g_next = *reinterpret_cast<const floatx4*>(norm.g + fin_n);
  }
  floatx4 cosv = floatx4{0.f, 0.f, 0.f, 0.f}, sinv = floatx4{0.f, 0.f, 0.f, 0.f};
  int qkv_page = 0;
  if constexpr (MODE == SK_QKV_ROPE) {
    if (wave == 0 && i < M) {
      if (qkv_head < rope.H + rope.Hk) {
        const float* cs = rope.cos_sin + (size_t)qkv_pos * rope.d;
        cosv = *reinterpret_cast<const floatx4*>(cs + qkv_e);
        sinv = *reinterpret_cast<const floatx4*>(cs + rope.d / 2 + qkv_e);
      }
      if (qkv_head >= rope.H) qkv_page = rope.block_table[(size_t)qkv_seg * rope.max_blocks + qkv_pos / rope.P];
    }
  }
  if (nsteps > 0) {
    int at = c_lo, done = 0;
    while (done + 3 < nsteps) {  // steps done, done+1 are loaded; done+2, done+3 exist
      compute(r0);
      load_step(r0, at + 2 * U);
      compute(r1);
      load_step(r1, at + 3 * U);
      at += 2 * U;
      done += 2;
    }
    const int rem = nsteps - done;  // 1..3
    compute(r0);
    if (rem == 3) load_step(r0, at + 2 * U);
    if (rem >= 2) compute(r1);
    if (rem == 3) compute(r0);
  }
  // Both tiles' sums of a row, in the lane i of the row
  floatx4 row[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    row[b] = acc[b][0][0] + eight_lanes_on(acc[b][0][1]);
    if constexpr (MG == 2) {
      const floatx4 second = eight_lanes_on(acc[b][1][0]) + acc[b][1][1];
      if (i >= 8) row[b] = second;
    }
  }
  // what is left of the range: single tiles, row i in the lanes i; the last one may be cut by K (K is a multiple of 8, so
  // a lane's 16 bytes of activations are inside or outside as a whole; W is zero beyond K)
  if (c_lo + nsteps * U < c_hi) {
    const bf16_t* rest = A + (size_t)min(i, M - 1) * lda + c * 8;
    for (int ch = c_lo + nsteps * U; ch < c_hi; ++ch) {
      const Frag af = ch * 32 + c * 8 < K ? load_frag(rest + ch * 32) : zero_frag();
#pragma unroll
      for (int b = 0; b < NB; ++b) row[b] = mfma16(load_frag_once(wb[b] + (size_t)ch * TILE_ELEMS), af, row[b]);
    }
  }

  if constexpr (PRE) {
    if constexpr (MG == 2) {
      ss_add(ss_v[0], 0), ss_add(ss_v[1], 1);
#pragma unroll 1
      for (int j = 2; j * WPB * 4 < ss_groups; ++j) ss_add(ss_load(j), j);   // more bands than 32 a wave
    }
    ss_piece += __shfl_xor(ss_piece, 16);
    ss_piece += __shfl_xor(ss_piece, 32);
    if (c == 0) row_ss[wave * 16 + i] = ss_piece;
  }
  // partial sums of the waves, added in wave order
  float* mine = red + wave * (NB * 256);
#pragma unroll
  for (int b = 0; b < NB; ++b) *reinterpret_cast<floatx4*>(&mine[(b * 64 + lane) * 4]) = row[b];
  __syncthreads();

  constexpr int NSUM = (MODE == SK_SWIGLU || MODE == SK_QKV_ROPE) ? 2 : 1;
  if (wave < ITEMS) {
    const int b = wave;
    floatx4 sum[NSUM];
#pragma unroll
    for (int s = 0; s < NSUM; ++s) {
      const int bb = NSUM == 2 ? s : b;
      sum[s] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WPB; ++w)
        sum[s] += *reinterpret_cast<const floatx4*>(&red[w * (NB * 256) + (bb * 64 + lane) * 4]);
    }
    const int m = i;  // D[n][m]: this lane holds row m = lane % 16 of the tile and columns fin_n .. fin_n + 3
    if constexpr (PRE) {
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < WPB; ++w) total += row_ss[w * 16 + i];
      const float rstd = 1.0f / sqrtf(total / (float)K + norm.eps);
#pragma unroll
      for (int s2 = 0; s2 < NSUM; ++s2) sum[s2] *= rstd;
    }
    if constexpr (MODE == SK_QKV_ROPE) {
      if (m < M) {
        float lo[4], hi[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          lo[r] = bf16_to_float(float_to_bf16(sum[0][r]));
          hi[r] = bf16_to_float(float_to_bf16(sum[1][r]));
        }
        const int half = rope.d / 2, slot = qkv_pos % rope.P;
        bf16_t* page = rope.cache + (size_t)qkv_page * ((size_t)2 * rope.Hk * rope.P * rope.d);
        if (qkv_head < rope.H + rope.Hk) {
          float ya[4], yb[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float av = lo[r], bv = hi[r], cc = cosv[r], sn = sinv[r];
            ya[r] = av * cc - bv * sn;
            yb[r] = av * sn + bv * cc;
          }
          bf16_t* dst = qkv_head < rope.H ? (bf16_t*)C + (size_t)m * ldc + (size_t)qkv_head * rope.d
                                          : page + ((size_t)(qkv_head - rope.H) * rope.P + slot) * rope.d;
          uint2 pa, pb;
          pa.x = pack_bf16x2(ya[0], ya[1]);
          pa.y = pack_bf16x2(ya[2], ya[3]);
          pb.x = pack_bf16x2(yb[0], yb[1]);
          pb.y = pack_bf16x2(yb[2], yb[3]);
          *reinterpret_cast<uint2*>(dst + qkv_e) = pa;
          *reinterpret_cast<uint2*>(dst + qkv_e + half) = pb;
        } else {
          bf16_t* col = page + (size_t)rope.Hk * rope.P * rope.d +
                        ((size_t)(qkv_head - rope.H - rope.Hk) * rope.d + qkv_e) * rope.P + slot;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            col[(size_t)r * rope.P] = float_to_bf16(sum[0][r]);
            col[(size_t)(half + r) * rope.P] = float_to_bf16(sum[1][r]);
          }
        }
      }
      return;
    }
    float sq = 0.f;  // EMIT: x^2 over this lane's columns
    if (fin_vec) {
      if (MODE == SK_STORE_BF16 || MODE == SK_SWIGLU || MODE == SK_ACT) {
        floatx4 y = sum[0];
        if (MODE == SK_ACT) {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = activation_f(sum[0][r], norm.act);
        }
        if (MODE == SK_SWIGLU) {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = silu_f(sum[0][r]) * sum[NSUM - 1][r];
        }
        uint2 packed;
        packed.x = pack_bf16x2(y[0], y[1]);
        packed.y = pack_bf16x2(y[2], y[3]);
        *reinterpret_cast<uint2*>((bf16_t*)C + (size_t)m * ldc + fin_n) = packed;
      } else if (MODE == SK_STORE_F32) {
        *reinterpret_cast<floatx4*>((float*)C + (size_t)m * ldc + fin_n) = sum[0];
      } else {
        const floatx4 x = c_old + sum[0];
        *reinterpret_cast<floatx4*>((float*)C + (size_t)m * ldc + fin_n) = x;
        if constexpr (EMIT) {
          uint2 packed;
          packed.x = pack_bf16x2(x[0] * g_next[0], x[1] * g_next[1]);
          packed.y = pack_bf16x2(x[2] * g_next[2], x[3] * g_next[3]);
          *reinterpret_cast<uint2*>(norm.raw + (size_t)m * norm.ld_raw + fin_n) = packed;
#pragma unroll
          for (int r = 0; r < 4; ++r) sq = fmaf(x[r], x[r], sq);
        }
      }
    } else if (m < M) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = fin_n + r;
        if (n >= N) continue;
        const size_t o = (size_t)m * ldc + n;
        if (MODE == SK_STORE_BF16) ((bf16_t*)C)[o] = float_to_bf16(sum[0][r]);
        else if (MODE == SK_ACT) ((bf16_t*)C)[o] = float_to_bf16(activation_f(sum[0][r], norm.act));
        else if (MODE == SK_STORE_F32) ((float*)C)[o] = sum[0][r];
        else if (MODE == SK_ACC_F32) {
          const float x = ((float*)C)[o] + sum[0][r];
          ((float*)C)[o] = x;
          if constexpr (EMIT) {
            norm.raw[(size_t)m * norm.ld_raw + n] = float_to_bf16(x * norm.g[n]);
            sq = fmaf(x, x, sq);
          }
        } else ((bf16_t*)C)[o] = float_to_bf16(silu_f(sum[0][r]) * sum[NSUM - 1][r]);
      }
    }
    if constexpr (EMIT) {  // the four lanes with pieces of row i add up (all lanes of the wave take part)
      sq += __shfl_xor(sq, 16);
      sq += __shfl_xor(sq, 32);
      if (c == 0 && band0 + b < bands) norm.ss[(size_t)i * norm.ld_ss + band0 + b] = sq;
    }
  }
}

// bands per block and waves per block: enough blocks and waves to keep HBM busy, never more waves than K
// can feed with whole steps or LDS can hold.  The waves, and with them the order of additions, do not depend on M.
// Of many bands a block takes two, one set of activations for both.  A K of 4,096, 8,192, .. puts a wave's two streams a power of
// two of 128 KiB and more apart, where they come at 6 TB/s instead of 7; one band a block then, while the activations are few.
// 128,256 outputs, one band / two, us: K 4,096 with 1, 8, 16 rows 155, 158, 188 / 177, 178, 182, K 8,192 305, 310, 368 / 345, 346,
// 354; 32,768 outputs, K 4,096, 8 rows 40 / 50; K 2,048, 8 rows 80 / 81, K 5,120 196 / 189, K 12,288 467 / 462.
static void pick_shape(int M, int N, int K, bool swiglu, int* nb, int* wpb) {
  const int bands = ceil_div(N, 16), chunks = ceil_div(K, 32);
  const bool streams_collide = chunks >= 128 && (chunks & (chunks - 1)) == 0;
  *nb = (!swiglu && bands >= 2048) && !(streams_collide && M <= 8) ? 2 : 1;
  const int blocks = ceil_div(bands, *nb);
  const int sets = swiglu ? 2 : *nb;
  int w = 4;
  while (w < 16 && (long)blocks * w < 4096 && chunks >= w * 2 * SK_U && w * 2 * sets <= 64) w *= 2;
  *wpb = w;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

template <int MODE, bool PRE, bool EMIT>
static int launch_skinny(const bf16_t* A, int lda, const bf16_t* W, const bf16_t* W2, void* C, int ldc, int M, int N,
                         int K, SkNorm norm, hipStream_t stream, SkRope rope = SkRope{}) {
  int nb, wpb;
  pick_shape(M, MODE == SK_QKV_ROPE ? N / 2 : N, K, MODE == SK_SWIGLU || MODE == SK_QKV_ROPE, &nb, &wpb);
  const int chunks = ceil_div(K, 32), bands = ceil_div(N, 16);
  if ((MODE == SK_SWIGLU || MODE == SK_QKV_ROPE) && wpb > 8) wpb = 8;
  if (PRE && norm.ld_ss > 4 * 4 * wpb * SS_LOADS) return APC_ERR_UNSUPPORTED;
  // whole 16-byte (float32) or 8-byte (bfloat16) accesses to C and to the emitted row where everything is aligned
  const int elem = (MODE == SK_STORE_BF16 || MODE == SK_SWIGLU || MODE == SK_ACT) ? 2 : 4;
  int vec_c = ldc % 4 == 0 && ((uintptr_t)C % (4 * elem)) == 0;
  if (EMIT) vec_c = vec_c && norm.ld_raw % 4 == 0 && ((uintptr_t)norm.raw % 8) == 0 && aligned16(norm.g);
#define SK_LAUNCH(NB_, WPB_)                                                                                  \
  hipLaunchKernelGGL((M <= 8 ? skinny_gemm_kernel<1, MODE, NB_, WPB_, PRE, EMIT>                              \
                             : skinny_gemm_kernel<2, MODE, NB_, WPB_, PRE, EMIT>),                            \
                     dim3(ceil_div(bands, MODE == SK_SWIGLU ? 1 : NB_)), dim3(WPB_ * WAVE), 0, stream, A, lda, W, \
                     W2, chunks, C, ldc, M, N, K, norm, vec_c, rope)
  if constexpr (MODE == SK_SWIGLU || MODE == SK_QKV_ROPE) {
    // two bands a wave: with 16 waves a block the two register sets of loads would not fit the 128 registers a
    // wave has then
    if (wpb == 4) SK_LAUNCH(2, 4);
    else SK_LAUNCH(2, 8);
  } else if (nb == 2) {
    if (wpb == 4) SK_LAUNCH(2, 4);
    else SK_LAUNCH(2, 8);
  } else {
    if (wpb == 4) SK_LAUNCH(1, 4);
    else if (wpb == 8) SK_LAUNCH(1, 8);
    else SK_LAUNCH(1, 16);
  }
#undef SK_LAUNCH
  APC_LAUNCH_CHECK();
  return 0;
}

static bool operands_ok(const void* A, int lda, const void* W, int M, int K) {
  return M <= 16 && K % 8 == 0 && lda % 8 == 0 && aligned16(A) && aligned16(W);
}

// W: tiled layout of an [N, K] matrix.  mode: 0 store bfloat16, 1 store float32, 2 add into float32, 17 .. 19: an
// activation (see activation_f; 16 + its code) on the sums, then store bfloat16
APC_EXPORT int apc_skinny_gemm_bf16(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                                    int mode, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N) return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, W, M, K)) return APC_ERR_UNSUPPORTED;
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  SkNorm none{};
  if (mode_is_act(mode)) {
    none.act = mode - MODE_ACT;
    return launch_skinny<SK_ACT, false, false>(a, lda, w, nullptr, C, ldc, M, N, K, none, stream);
  }
  switch (mode) {
    case SK_STORE_BF16: return launch_skinny<SK_STORE_BF16, false, false>(a, lda, w, nullptr, C, ldc, M, N, K, none, stream);
    case SK_STORE_F32: return launch_skinny<SK_STORE_F32, false, false>(a, lda, w, nullptr, C, ldc, M, N, K, none, stream);
    case SK_ACC_F32: return launch_skinny<SK_ACC_F32, false, false>(a, lda, w, nullptr, C, ldc, M, N, K, none, stream);
    default: return APC_ERR_BAD_ARG;
  }
}

// out[m, f] = silu(A[m] . Wg[f]) * (A[m] . Wu[f]);  Wg, Wu: tiled layouts of two [F, K] matrices
APC_EXPORT int apc_skinny_swiglu_bf16(const void* A, int lda, const void* Wg, const void* Wu, void* C, int ldc, int M,
                                      int F, int K, hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if (K <= 0 || lda < K || ldc < F) return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, Wg, M, K) || !aligned16(Wu)) return APC_ERR_UNSUPPORTED;
  return launch_skinny<SK_SWIGLU, false, false>((const bf16_t*)A, lda, (const bf16_t*)Wg, (const bf16_t*)Wu, C, ldc, M,
                                                F, K, SkNorm{}, stream);
}

// C += A . W^T into the float32 residual C [M, N], and for the RMS norm that reads C next: raw[m, n] =
// bfloat16(C[m, n] * g[n]) and ss[row][band] = the sum of C^2 over the band's 16 columns (ss: 16 rows of
// ceil(N / 16) floats rounded up to a multiple of 4).
APC_EXPORT int apc_skinny_gemm_emit_bf16(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                                         const float* g, void* raw, int ld_raw, float* ss, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N || ld_raw < N || !g || !raw || !ss) return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, W, M, K)) return APC_ERR_UNSUPPORTED;
  const SkNorm norm{ss, ceil_div(N, 16), ceil_div(ceil_div(N, 16), 4) * 4, 0.f, g, (bf16_t*)raw, ld_raw};
  return launch_skinny<SK_ACC_F32, false, true>((const bf16_t*)A, lda, (const bf16_t*)W, nullptr, C, ldc, M, N, K, norm,
                                                stream);
}

// The two storing products on a row that apc_skinny_gemm_emit_bf16 left: A = raw [M, K], ss = [16][n_ss rounded up
// to 4] sums of x^2 (n_ss = ceil(K / 16)); out = (A . W^T) / sqrt(sum(ss) / K + eps).  mode: 0 store bfloat16, 1 store float32.
APC_EXPORT int apc_skinny_gemm_pre_bf16(const void* A, int lda, const float* ss, int n_ss, float eps, const void* W,
                                        void* C, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N || !ss || n_ss <= 0 || !aligned16(ss)) return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, W, M, K)) return APC_ERR_UNSUPPORTED;
  const SkNorm norm{const_cast<float*>(ss), n_ss, ceil_div(n_ss, 4) * 4, eps, nullptr, nullptr, 0};
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  switch (mode) {
    case SK_STORE_BF16: return launch_skinny<SK_STORE_BF16, true, false>(a, lda, w, nullptr, C, ldc, M, N, K, norm, stream);
    case SK_STORE_F32: return launch_skinny<SK_STORE_F32, true, false>(a, lda, w, nullptr, C, ldc, M, N, K, norm, stream);
    default: return APC_ERR_BAD_ARG;
  }
}

APC_EXPORT int apc_skinny_swiglu_pre_bf16(const void* A, int lda, const float* ss, int n_ss, float eps, const void* Wg,
                                          const void* Wu, void* C, int ldc, int M, int F, int K, hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if (K <= 0 || lda < K || ldc < F || !ss || n_ss <= 0 || !aligned16(ss)) return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, Wg, M, K) || !aligned16(Wu)) return APC_ERR_UNSUPPORTED;
  const SkNorm norm{const_cast<float*>(ss), n_ss, ceil_div(n_ss, 4) * 4, eps, nullptr, nullptr, 0};
  return launch_skinny<SK_SWIGLU, true, false>((const bf16_t*)A, lda, (const bf16_t*)Wg, (const bf16_t*)Wu, C, ldc, M, F,
                                               K, norm, stream);
}

// q, k, v of M <= 16 rows in one product, q and k rotated, k and v written into the paged cache (see SkRope).
// W: tiled layout of [(H + 2 Hk) d, K]; q_out [M, ldq] takes the rotated q heads in its first H d columns.  With ss:
// A is a row that apc_skinny_gemm_emit_bf16 left and the sums are scaled as in apc_skinny_gemm_pre_bf16.
APC_EXPORT int apc_skinny_qkv_rope_bf16(const void* A, int lda, const float* ss, int n_ss, float eps, const void* W,
                                        void* q_out, int ldq, int M, int K, int H, int Hk, int d,
                                        const float* cos_sin, const int* positions, const int* row_seg,
                                        const int* block_table, int max_blocks, void* cache, int page_tokens,
                                        hipStream_t stream) {
  if (M <= 0) return 0;
  if (H <= 0 || Hk <= 0 || d <= 0 || K <= 0 || lda < K || ldq < H * d || !cos_sin || !positions || !row_seg ||
      !block_table || max_blocks <= 0 || !cache || page_tokens <= 0 || (ss && n_ss <= 0))
    return APC_ERR_BAD_ARG;
  if (!operands_ok(A, lda, W, M, K) || d % 32 || ldq % 4 || ((uintptr_t)q_out & 7u) || !aligned16(cos_sin) ||
      ((uintptr_t)cache & 7u) || (ss && !aligned16(ss)))
    return APC_ERR_UNSUPPORTED;
  const SkRope rope{cos_sin, positions, row_seg, block_table, max_blocks, (bf16_t*)cache, page_tokens, H, Hk, d};
  const int N = (H + 2 * Hk) * d;
  if (ss) {
    const SkNorm norm{const_cast<float*>(ss), n_ss, ceil_div(n_ss, 4) * 4, eps, nullptr, nullptr, 0};
    return launch_skinny<SK_QKV_ROPE, true, false>((const bf16_t*)A, lda, (const bf16_t*)W, nullptr, q_out, ldq, M, N, K,
                                                   norm, stream, rope);
  }
  return launch_skinny<SK_QKV_ROPE, false, false>((const bf16_t*)A, lda, (const bf16_t*)W, nullptr, q_out, ldq, M, N, K,
                                                  SkNorm{}, stream, rope);
}
