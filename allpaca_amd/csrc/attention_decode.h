// Attention of decoded rows (one row a request) over the paged cache in bfloat16: the work of a block, for the kernels of
// attention_bf16.hip and for the kernel of attention_wide_bf16.hip that runs it beside tiles of prompt rows.
#pragma once
#include "mfma.h"
#include <math.h>

namespace attn_decode {

constexpr int KPAD = 8;

__device__ __forceinline__ float row4_max(float v) {  // over the 4 lanes that share lane % 16
  v = fmaxf(v, __shfl_xor(v, 16, WAVE));
  return fmaxf(v, __shfl_xor(v, 32, WAVE));
}
__device__ __forceinline__ float row4_sum(float v) {
  v += __shfl_xor(v, 16, WAVE);
  return v + __shfl_xor(v, 32, WAVE);
}
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) { return pack_bf16x2(a, b); }
// A value operand holds 8 consecutive positions of one element.  Positions beyond the row's last key lie in slots
// that nobody has written since the page's last owner, positions in front of a window's first key may lie in the
// spare page that stands in for pages given back.  Their weight in P is 0, but 0 x NaN is NaN, so all but the
// positions lo <= p < hi of the 8 are cleared before the product sees them.
__device__ __forceinline__ void keep_positions(Frag& v, int lo, int hi) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t a = (2 * w >= lo && 2 * w < hi) ? 0x0000ffffu : 0u;
    const uint32_t b = (2 * w + 1 >= lo && 2 * w + 1 < hi) ? 0xffff0000u : 0u;
    v.w[w] &= a | b;
  }
}
// 2^x for x <= 0 (or -inf): the bare instruction, without the range handling that large arguments need
__device__ __forceinline__ float exp2_neg(float x) { return __builtin_amdgcn_exp2f(x); }
constexpr float LOG2E = 1.4426950408889634f;

// parts[row][head][part][d + 2]: o[0..d), m, l
template <int DP>
struct KVRegs {
  Frag k[2][DP / 32];  // two tiles of 16 keys
  Frag v[DP / 16];     // 32 positions of 16 value elements per tile
};

// Two loads of keys as they come, 8 keys x 64 elements each (lane: key lane % 8, 16 bytes (lane % 16 / 8) * 4 + lane / 16 of
// the 128 of its line), into two operands of 16 keys x 32 elements: the lanes 8-15 of 16 of the first load change places with the
// lanes 0-7 of the second.
__device__ __forceinline__ void lines_to_operands(Frag& a, Frag& b) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int x = (int)a.w[w], y = (int)b.w[w];
    a.w[w] = (uint32_t)__builtin_amdgcn_update_dpp(x, y, 0x128, 0xf, 0xc, false);   // row_ror:8 into the lanes 8-15
    b.w[w] = (uint32_t)__builtin_amdgcn_update_dpp(y, x, 0x128, 0xf, 0x3, false);   // and into the lanes 0-7
  }
}

// Ways to the finished heads of a (row, kv head):
//  DEC_PARTS  a block is 4 parts (ranges of KW keys) of the pair; its waves leave their results in `parts` and
//             attn_merge_kernel, a second launch, finishes.  Kept for the sizes the other two do not take.
//  DEC_LAST   the same split over blocks, but a block first adds its 4 waves' results in LDS, leaves ONE partial
//             result, and the block of a pair that finishes last adds the blocks' results in block order and writes
//             the heads: no second launch (4.7-5.6 us a layer at 8B shapes, as much as the attention itself with one
//             row).  Who is last is found with one counter per pair (a block adds 1 when its result is in memory;
//             the one that reads blocks - 1 is last, and sets the counter back to 0 for the next launch).  The
//             partial results go through memory with stores and loads that are coherent across the chip's eight L2
//             caches one by one (sc1), not with a fence: a device-wide fence writes back and invalidates a whole L2
//             and cost ten times what the second launch did.
//  DEC_WHOLE  the block's 4 waves take all ranges of KW keys of the pair in turn (wave w the ranges w, w + 4, ..; with
//             KW == 0 the row's own keys in 4 equal ranges, one a wave, so that a short row beside a long one still
//             has work for every wave: 32 rows of 328 to 4,296 keys 69.1 -> 66.7 us, equal rows as before),
//             meet in LDS and the block writes the finished heads itself: no partial result goes through memory,
//             which pays once the pairs alone fill the chip (8B shapes, 2,048 keys a row: 32 rows 52.9 -> 49.1 us, 64
//             rows 98.2 -> 91.6 us, 128 rows 196 -> 181 us; with 16 rows 30.2 -> 34.7 us.  Blocks of 8 waves were 2 %
//             faster at one block a compute unit and 8-15 % slower at two).
//  DEC_EVEN   rows of very different lengths, where a block a pair leaves the chip waiting for the longest row's block (64
//             rows of 90 to 2,100 keys: 63 us of which the bytes are 23).  Each kv head's work, the steps of 32 keys of
//             all its rows one after the other (a row counts two steps more for what it costs beside its keys), goes in
//             equal shares to the waves of one round of blocks; every wave finds its share and the rows it falls into
//             from the rows' positions, so a recorded graph fits whatever lengths they reach.  A row inside one share is
//             finished by its wave; the pieces of a row that lies in several go through memory as in DEC_LAST, and the
//             wave that leaves the last of them adds them in order.  37 us there.  What is left over the bytes is a
//             wave's chain of rows, about 4 us each, and the way of the pieces through memory, so rows of about one
//             length are better off with DEC_WHOLE (32 rows of 1,100 keys on 8 kv heads of 128: 26.1 and 31.8 us): the
//             caller chooses by the lengths.  Choosing inside the kernel was slower both ways: the registers of either
//             path cost the other a wave a SIMD at heads of 64 (96 rows 53.8 -> 61.8 us), and a look at all rows
//             1 to 4 us.
// The order of additions for a row depends on its position, KW and the number of parts only (DEC_EVEN: on the lengths of
// the rows in front of it too).
// LINES (heads of 64 and 128, pages of a power of two): a load of keys asks for 8 whole lines of 128 bytes instead of 16 half
// ones, and 24 moves between the lanes of a row of 16 a 16 keys of a head of 128 make operands of two such loads; the page
// of a group of 8 keys is one value for the wave, so places are scalar work and no look-up goes through LDS.  What bounds
// the kernel beside its bytes is the chain to the first keys and what a unit's loads cost (half lines leave the L2 at a third of
// the rate).  One layer, 32 heads over 8, without / with, us: heads of 128, 1 row x 387 keys 10.8 / 10.1, 8 x 2,048 18.0 / 17.1,
// 64 x 100 12.5 / 9.5, 64 x 1,000 50.2 / 46.0, 64 rows of 90 to 2,100 (DEC_EVEN) 39.3 / 36.1; heads of 64, 1 x 387 8.0 / 7.4, 8 x 2,048
// 11.8 / 11.3, 64 x 2,048 47.9 / 46.7.  Of 1,791 sizes (1 to 256 rows of 1 to 8,192 keys, six pairs of heads), 0.94 in the mean, rows of up
// to 31 keys are 0.1 us slower, and 384 to 768 (row, kv head) pairs of heads of 64 with up to 64 keys 0.2 of 5 us: three and four blocks
// fit on a unit instead of three, and are not spread as evenly.  The same bits.
constexpr int NW = 4;  // waves of a block of the decode kernel
constexpr int LAST_DIRECT = 8;  // up to so many blocks a pair the last one reads the others' results in one go
enum { DEC_PARTS = 0, DEC_WHOLE = 1, DEC_LAST = 2, DEC_EVEN = 3 };
// Keys a part of a row takes when the launch gives the number of parts and not their length (KW == 0): the row's
// `span` keys in n_parts equal ranges, in whole steps of 32 keys and no fewer than 64.  Rows of different lengths in
// one launch then all use every block of their pair, and a launch's shape (blocks a pair) does not change with the
// rows' lengths, which is what a recorded graph needs.
__device__ __forceinline__ int row_keys_per_part(int KW, int span, int n_parts) {
  if (KW > 0) return KW;
  return max(64, ((span + n_parts - 1) / n_parts + 31) / 32 * 32);
}
// Why the hand-over of DEC_LAST holds without a release/acquire pair.  Every access to a partial result, on either
// side, is a relaxed atomic of agent scope: on this chip such a store goes through to memory past the block's own L2
// (sc1) and such a load is served from memory, so neither a write-back of the writer's L2 nor an invalidation of the
// reader's is needed for these words.  What is left is order: a writer thread's stores are issued before its
// `s_waitcnt vmcnt(0)`, which returns when memory has acknowledged them; the block's barrier behind it puts all its
// threads' acknowledged stores before thread 0's add to the counter; the counter's adds are atomics on one word, so the
// block that reads `nz - 1` adds after every other block's add, hence after their stores were acknowledged; its
// loads are issued behind its own barrier, which stands behind that add.  The language's memory model does not
// promise this for relaxed atomics; the instructions they compile to here do (the kernel is built for gfx950 alone).
// The counters are zero before the first launch and every launch leaves them zero; a launch that dies half-way
// would leave a count behind, so whoever owns them zeroes them when an engine is set up (engine/native.py).
__device__ __forceinline__ void st_coh(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_coh(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same accesses (sc1, as the two above compile to), 16 and 8 bytes at a time; places in floats.
constexpr int COHERENT = 16;
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st_coh4(BufferRsrc to, int place, floatx4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), to, 4 * place, 0, COHERENT);
}
__device__ __forceinline__ floatx4 ld_coh4(BufferRsrc from, int place) {
  return __builtin_bit_cast(floatx4, (u32x4_t)__builtin_amdgcn_raw_buffer_load_b128(from, 4 * place, 0, COHERENT));
}
__device__ __forceinline__ floatx2 ld_coh2(BufferRsrc from, int place) {
  return __builtin_bit_cast(floatx2, (u32x2_t)__builtin_amdgcn_raw_buffer_load_b64(from, 4 * place, 0, COHERENT));
}
__device__ __forceinline__ int wave_sum_int(int v) {
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
  return v;
}
__device__ __forceinline__ int wave_scan_int(int v) {  // the sum of this lane's and all earlier lanes' values
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const int up = __shfl_up(v, o, WAVE);
    if ((int)(threadIdx.x % WAVE) >= o) v += up;
  }
  return v;
}
// DEC_EVEN: what a row costs beside its steps of 32 keys (page ids, query, the first loads' way, its result), in steps,
// and the least that a wave is given.
// EVEN_BLOCKS: a block a compute unit (two, where registers allow them, were slower: 64 ragged rows 37 -> 48 us, more
// pieces and as many bytes in flight).  EVEN_BATCH: pieces of a row that the last wave asks for together.
constexpr int EVEN_ROW_COST = 2, EVEN_MIN_SHARE = 8, EVEN_BLOCKS = 256, EVEN_BATCH = 4;
// Where the pieces of kv head tile `tile` lie in the workspace, in floats: a region for every tile, two places a wave.
// All regions have the room of a full tile: blocks of all tiles run side by side, and the last tile of a group may have
// fewer heads than the others.
struct EvenRoom {
  int tile_heads, stride;  // heads of the tile; a head of a piece: its sums, maximum, sum, room
  long long first, end;
};
__host__ __device__ inline EvenRoom even_room(int G, int d, int waves, int tile) {
  const int left = G - tile % ((G + 15) / 16) * 16, heads = left < 16 ? left : 16;
  const long long place = (long long)waves * 2 * (d + 4), first = tile * place * (G < 16 ? G : 16);
  return {heads, d + 4, first, first + place * heads};
}
// Where a block stands in a launch of blocks (rows; kv heads and their tiles of 16 heads; ranges of keys)
struct DecodeAt {
  int row, pair, range, rows, pairs, ranges;
};
constexpr int DEC_P_ELEMS = NW * 16 * (32 + KPAD);   // a block's P of all waves, in LDS
// The work of a block.  Ps: DEC_P_ELEMS; meet: [NW][heads of the tile][d + 2] (DEC_WHOLE, DEC_LAST); is_last: DEC_LAST.
template <int DP, int MODE, bool LINES>
__device__ __forceinline__ void attn_decode_block(
    const DecodeAt blk, bf16_t* Ps, float* meet, int* is_last,
    const bf16_t* __restrict__ q, int ldq, int q_off, int H, int Hk, int d, const bf16_t* __restrict__ cache, int P,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ positions,
    const int* __restrict__ row_seg, const int* __restrict__ rows, int window, float scale, int KW, int n_parts,
    float* __restrict__ parts, bf16_t* __restrict__ out, int ldo, int* __restrict__ counters) {
  constexpr bool WHOLE = MODE == DEC_WHOLE, LAST = MODE == DEC_LAST, EVEN = MODE == DEC_EVEN;
  static_assert(!LINES || DP % 64 == 0, "whole lines of 64 elements");
  const int lane = threadIdx.x % WAVE, wave = LINES ? __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) : threadIdx.x / WAVE;
  const int li = lane % 16, lc = lane / 16;
  const int G = H / Hk, gtiles = (G + 15) / 16;
  const int ri = blk.row;
  const int kvh = blk.pair / gtiles, gt = blk.pair % gtiles;
  const int part = blk.range * NW + wave;
  int row = 0, pos = 0, first = 0, seen0 = 0;  // the row in work; seen0: the first position that is loaded
  const int* bt = nullptr;
  auto take_row = [&](int r, int position, int seg) {
    row = r;
    pos = position;
    first = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    seen0 = (first / 32) * 32;
    bt = block_table + (size_t)seg * max_blocks;
  };
  bool empty = false;
  int base = 0;
  if constexpr (!EVEN) {
    const int r = rows ? rows[ri] : ri;
    take_row(r, positions[r], row_seg[r]);
    // KW == 0: the row's own keys, from the first one it sees, in n_parts equal ranges (see row_keys_per_part); else
    // ranges of KW keys counted from position 0
    base = KW > 0 ? 0 : seen0;
    KW = row_keys_per_part(KW, pos + 1 - seen0, n_parts);
    // nothing to see for this part: the wave leaves (DEC_PARTS), or stays with an empty result (DEC_LAST: the block's
    // waves meet)
    empty = !WHOLE && (part >= n_parts || max(base + part * KW, seen0) >= min(base + (part + 1) * KW, pos + 1));
    if (MODE == DEC_PARTS && empty) return;
  }
  const size_t page_stride = (size_t)2 * Hk * P * d;
  const size_t head_off = (size_t)kvh * P * d, v_off = (size_t)Hk * P * d;
  // the page ids of a range of keys, one per lane, fetched once per range: the loads of keys and values then
  // do not wait for a look-up in the block table (a range of KW keys spans at most 64 pages: checked by the host)
  int page0 = 0, my_page = 0;

  Frag qf[DP / 32];
  floatx4 o[DP / 16];
  float m_run, l_run;
  auto begin_row = [&]() {
    const int g = gt * 16 + li;
    const bf16_t* qrow = q + (size_t)row * ldq + q_off + (size_t)(kvh * G + min(g, G - 1)) * d;
#pragma unroll
    for (int ks = 0; ks < DP / 32; ++ks) {
      const int e = ks * 32 + lc * 8;
      qf[ks] = (g < G && e < d) ? load_frag(qrow + e) : zero_frag();
    }
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    m_run = -INFINITY;
    l_run = 0.f;
  };
  if constexpr (!EVEN) begin_row();
  bf16_t* pw = Ps + wave * 16 * (32 + KPAD);

  // Operands of 32 keys straight from the pages, with loads that the caches do not keep (a decoded row reads its keys
  // and values once).  Nothing is loaded conditionally: a key beyond the row's own
  // position is read from that position instead (its score is masked), an element beyond d from element 0 or
  // d - 1 (the query is zero there; such output columns are not stored), so the loads of the next 32 keys can be
  // in flight while these are used.
  const int lgP = LINES ? 31 - __builtin_clz(P) : 0;
  auto load_kv = [&](KVRegs<DP>& r, int kb) {
    if constexpr (LINES) {
      const int last8 = pos & ~7;          // the group of 8 keys with the row's own: what lies beyond is read from there
      size_t at[4];                        // of the groups' keys 0 in the head's part of the cache
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int g0 = min(kb + 8 * h, last8), rr = min(li % 8, pos - g0);
        const int page = __builtin_amdgcn_readlane(my_page, (g0 >> lgP) - page0);
        at[h] = (size_t)page * page_stride + head_off;
        const bf16_t* krow = cache + at[h] + (size_t)(g0 & (P - 1)) * DP + (rr * DP + ((li / 8) * 4 + lc) * 8);
        at[h] += v_off + (g0 & (P - 1));
#pragma unroll
        for (int kp = 0; kp < DP / 64; ++kp) r.k[h / 2][2 * kp + h % 2] = load_frag_once(krow + kp * 64);
      }
      const size_t mine = lc == 0 ? at[0] : lc == 1 ? at[1] : lc == 2 ? at[2] : at[3];
      const bf16_t* vbase = cache + mine + (size_t)li * P;
#pragma unroll
      for (int dt = 0; dt < DP / 16; ++dt) r.v[dt] = load_frag_once(vbase + (size_t)dt * 16 * P);
      return;
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int t = min(kb + nt * 16 + li, pos);
      const int page = __shfl(my_page, t / P - page0, WAVE);
      const bf16_t* krow = cache + (size_t)page * page_stride + head_off + (size_t)(t % P) * d;
#pragma unroll
      for (int ks = 0; ks < DP / 32; ++ks) {
        const int e = ks * 32 + lc * 8;
        r.k[nt][ks] = load_frag_once(krow + (e < d ? e : 0));
      }
    }
    const int tv = min(kb + lc * 8, (pos / 8) * 8);
    const int vpage = __shfl(my_page, tv / P - page0, WAVE);
    const bf16_t* vbase = cache + (size_t)vpage * page_stride + v_off + head_off + (tv % P);
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt) r.v[dt] = load_frag_once(vbase + (size_t)min(dt * 16 + li, d - 1) * P);
  };

  // lane holds keys kb + nt*16 + lc*4 + r (scores) and elements dt*16 + lc*4 + r (output) of head li of the group
  const float sc2 = scale * LOG2E;
  auto step = [&](KVRegs<DP>& r, int kb) {
    if (kb + 31 > pos || kb < first) {  // a step with positions the row does not see (see keep_positions)
      const int tv = min(kb + lc * 8, (pos / 8) * 8);  // as load_kv placed this lane's 8 positions
      const int lo = first - tv, hi = pos - tv + 1;
      if (lo > 0 || hi < 8) {
#pragma unroll
        for (int dt = 0; dt < DP / 16; ++dt) keep_positions(r.v[dt], lo, hi);
      }
    }
    floatx4 s[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      s[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (LINES) {
#pragma unroll
        for (int kp = 0; kp < DP / 64; ++kp) lines_to_operands(r.k[nt][2 * kp], r.k[nt][2 * kp + 1]);
      }
#pragma unroll
      for (int ks = 0; ks < DP / 32; ++ks) s[nt] = mfma16(r.k[nt][ks], qf[ks], s[nt]);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int t = kb + nt * 16 + lc * 4 + rr;
        const float v = (t >= first && t <= pos) ? s[nt][rr] * sc2 : -INFINITY;
        s[nt][rr] = v;
        mx = fmaxf(mx, v);
      }
    mx = row4_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_neg(m_run - m_safe);
    float sum = 0.f;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const float pv = exp2_neg(s[nt][rr] - m_safe);
        s[nt][rr] = pv;
        sum += pv;
      }
      uint2 pk;
      pk.x = bf16_pair(s[nt][0], s[nt][1]);
      pk.y = bf16_pair(s[nt][2], s[nt][3]);
      *reinterpret_cast<uint2*>(&pw[li * (32 + KPAD) + nt * 16 + lc * 4]) = pk;
    }
    l_run = l_run * alpha + row4_sum(sum);
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) o[dt][rr] *= alpha;
    wave_lds_order();
    const Frag pf = *reinterpret_cast<const Frag*>(&pw[li * (32 + KPAD) + lc * 8]);
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt) o[dt] = mfma16(r.v[dt], pf, o[dt]);
    wave_lds_order();
  };

  auto run_range = [&](int k_lo, int k_hi) {
    page0 = LINES ? k_lo >> lgP : k_lo / P;
    my_page = bt[min(page0 + lane, LINES ? pos >> lgP : pos / P)];
    const int nsteps = (k_hi - k_lo + 31) / 32;
    KVRegs<DP> ra, rb;
    load_kv(ra, k_lo);
    int done = 0, kb = k_lo;
    while (done + 2 < nsteps) {
      load_kv(rb, kb + 32);
      step(ra, kb);
      load_kv(ra, kb + 64);
      step(rb, kb + 32);
      kb += 64;
      done += 2;
    }
    if (done + 1 < nsteps) {
      load_kv(rb, kb + 32);
      step(ra, kb);
      step(rb, kb + 32);
    } else {
      step(ra, kb);
    }
  };
  // a range in pieces of no more keys than a wave keeps page ids for (one piece, but for rows far longer than the
  // launch's parts were counted for, and for the one range a wave of DEC_WHOLE has of a long row)
  const int piece = max(32, (62 * P) / 32 * 32);
  if constexpr (EVEN) {
    // This wave's share of its kv head's work, and the rows it falls into.  Rows are looked at 64 at a time, one a lane.
    const int waves = blk.rows * NW, me = blk.row * NW + wave;
    int r_l = 0, pos_l = 0, seg_l = 0, cost_l = 0;
    auto look_at = [&](int i0) {
      cost_l = 0;
      const int i = i0 + lane;
      if (i >= n_parts) return;
      r_l = rows ? rows[i] : i;
      pos_l = positions[r_l];
      seg_l = row_seg[r_l];
      const int f = (window > 0 && pos_l - window + 1 > 0) ? pos_l - window + 1 : 0;
      cost_l = (pos_l - f / 32 * 32) / 32 + 1 + EVEN_ROW_COST;
    };
    look_at(0);
    int end_l = wave_scan_int(cost_l), total = __builtin_amdgcn_readlane(end_l, WAVE - 1);
    if (n_parts > WAVE) {
      for (int i0 = WAVE; i0 < n_parts; i0 += WAVE) {
        look_at(i0);
        total += wave_sum_int(cost_l);
      }
      look_at(0);
    }
    const int share = max(EVEN_MIN_SHARE, (total + waves - 1) / waves);
    const int lo = me * share, hi = min(lo + share, total);
    const EvenRoom room = even_room(G, d, waves, blk.pair);
    const int tile_heads = room.tile_heads, stride = room.stride;
    const BufferRsrc pieces = make_rsrc(parts + room.first);
    for (int i0 = 0;;) {
      const int start_l = end_l - cost_l;
      unsigned long long todo = __ballot(cost_l > 0 && end_l > lo && start_l < hi);
      const int before = __builtin_amdgcn_readlane(end_l, WAVE - 1);
      for (; todo; todo &= todo - 1) {
        const int l = __ffsll(todo) - 1;
        const int steps0 = __builtin_amdgcn_readlane(start_l, l) + EVEN_ROW_COST;   // where the row's steps begin
        const int steps = __builtin_amdgcn_readlane(end_l, l) - steps0;
        const int s_lo = max(lo - steps0, 0), s_hi = min(hi - steps0, steps);
        if (s_lo >= s_hi) continue;
        take_row(__builtin_amdgcn_readlane(r_l, l), __builtin_amdgcn_readlane(pos_l, l), __builtin_amdgcn_readlane(seg_l, l));
        begin_row();
        const int k_hi = min(seen0 + 32 * s_hi, pos + 1);
        for (int k = seen0 + 32 * s_lo; k < k_hi; k += piece) run_range(k, min(k + piece, k_hi));
        const int g = gt * 16 + li;
        const int w0 = steps0 / share, n_pieces = (steps0 + steps - 1) / share - w0 + 1;
        bf16_t* heads = out + (size_t)row * ldo + (size_t)(kvh * G + gt * 16) * d;
        if (n_pieces == 1) {
          if (g < G) {
#pragma unroll
            for (int dt = 0; dt < DP / 16; ++dt) {
              const int e = dt * 16 + lc * 4;
              if (e < d) {
                uint2 pk;
                pk.x = bf16_pair(o[dt][0] / l_run, o[dt][1] / l_run);
                pk.y = bf16_pair(o[dt][2] / l_run, o[dt][3] / l_run);
                *reinterpret_cast<uint2*>(heads + (size_t)li * d + e) = pk;
              }
            }
          }
          continue;
        }
        // one of several pieces: the row's first piece is its wave's last, in place 1; the others are their wave's first
        if (g < G) {
          const int at = ((2 * me + (s_lo == 0 ? 1 : 0)) * tile_heads + li) * stride;
#pragma unroll
          for (int dt = 0; dt < DP / 16; ++dt) {
            const int e = dt * 16 + lc * 4;
            if (e < d) st_coh4(pieces, at + e, o[dt]);
          }
          if (lc == 0) st_coh4(pieces, at + d, floatx4{m_run, l_run, 0.f, 0.f});
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's stores have reached memory
        int* counter = counters + (size_t)(i0 + l) * blk.pairs + blk.pair;
        int done = 0;
        if (lane == 0) done = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(done) != n_pieces - 1) continue;
        // the last of the row's waves: all pieces in order, some at a time
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
        const int quads = tile_heads * d / 4;
        for (int x0 = 0; x0 < quads; x0 += 2 * WAVE) {   // two quads of elements a lane
          floatx4 acc[2];
          float m[2], sum[2];
          int at[2], last[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int x = min(x0 + u * WAVE + lane, quads - 1), hg = 4 * x / d;
            at[u] = (2 * w0 * tile_heads + hg) * stride + 4 * x - hg * d;
            last[u] = (2 * w0 * tile_heads + hg) * stride + d;
            acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
            m[u] = -INFINITY;
            sum[u] = 0.f;
          }
          for (int p0 = 0; p0 < n_pieces; p0 += EVEN_BATCH) {
            floatx4 po[2][EVEN_BATCH];
            floatx2 ml[2][EVEN_BATCH];
#pragma unroll
            for (int p = 0; p < EVEN_BATCH; ++p)
#pragma unroll
              for (int u = 0; u < 2; ++u) {
                const int pp = min(p0 + p, n_pieces - 1), off = (2 * pp + (pp == 0 ? 1 : 0)) * tile_heads * stride;
                ml[u][p] = ld_coh2(pieces, last[u] + off);
                po[u][p] = ld_coh4(pieces, at[u] + off);
              }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              float m_new = m[u];
#pragma unroll
              for (int p = 0; p < EVEN_BATCH; ++p)
                if (p0 + p < n_pieces) m_new = fmaxf(m_new, ml[u][p][0]);
              const float m_safe = m_new == -INFINITY ? 0.f : m_new, old = exp2_neg(m[u] - m_safe);
              m[u] = m_new;
              sum[u] *= old;
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[u][r] *= old;
#pragma unroll
              for (int p = 0; p < EVEN_BATCH; ++p)
                if (p0 + p < n_pieces) {
                  const float wgt = exp2_neg(ml[u][p][0] - m_safe);
                  sum[u] = fmaf(ml[u][p][1], wgt, sum[u]);
#pragma unroll
                  for (int r = 0; r < 4; ++r) acc[u][r] = fmaf(po[u][p][r], wgt, acc[u][r]);
                }
            }
          }
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int x = x0 + u * WAVE + lane;
            if (x >= quads) continue;
            uint2 pk;
            pk.x = bf16_pair(acc[u][0] / sum[u], acc[u][1] / sum[u]);
            pk.y = bf16_pair(acc[u][2] / sum[u], acc[u][3] / sum[u]);
            *reinterpret_cast<uint2*>(heads + 4 * x) = pk;
          }
        }
      }
      i0 += WAVE;
      if (i0 >= n_parts || before >= hi) return;
      look_at(i0);
      end_l = before + wave_scan_int(cost_l);
    }
  }
  if constexpr (WHOLE) {
    // ranges wave, wave + NW, ..: with the row's own ranges (the launch gave no length) that is one range a wave
    for (int r = wave; base + r * KW <= pos; r += NW) {
      const int k_lo = max(base + r * KW, seen0), k_hi = min(base + (r + 1) * KW, pos + 1);
      for (int k = k_lo; k < k_hi; k += piece) run_range(k, min(k + piece, k_hi));
    }
  } else if (!empty) {
    const int k_lo = max(base + part * KW, seen0), k_hi = min(base + (part + 1) * KW, pos + 1);
    for (int k = k_lo; k < k_hi; k += piece) run_range(k, min(k + piece, k_hi));
  }

  // this wave's result for the heads of the group (maxima are in base-2 units, as the merge expects)
  const int g = gt * 16 + li;
  const int tile_heads = min(G - gt * 16, 16);
  if (g < G) {
    float* dst = (WHOLE || LAST) ? meet + ((size_t)wave * tile_heads + li) * (d + 2)
                                 : parts + (((size_t)ri * H + (kvh * G + g)) * n_parts + part) * (d + 2);
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt) {
      const int e = dt * 16 + lc * 4;
      if (e < d) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) dst[e + rr] = o[dt][rr];
      }
    }
    if (lc == 0) { dst[d] = m_run; dst[d + 1] = l_run; }
  }
  if constexpr (WHOLE) {
    // the waves' results of a head, in wave order (a wave that saw no key left a maximum of -inf and zeros)
    __syncthreads();
    const int stride = d + 2;
    for (int idx = threadIdx.x; idx < tile_heads * d; idx += NW * 64) {
      const int hg = idx / d, e = idx % d;
      const float* src = meet + (size_t)hg * stride;
      float m = -INFINITY;
#pragma unroll
      for (int w = 0; w < NW; ++w) m = fmaxf(m, src[(size_t)w * tile_heads * stride + d]);
      float l = 0.f, acc = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float* ws = src + (size_t)w * tile_heads * stride;
        const float pm = ws[d];
        const float wgt = pm == -INFINITY ? 0.f : exp2_neg(pm - m);
        l += ws[d + 1] * wgt;
        acc = fmaf(ws[e], wgt, acc);
      }
      out[(size_t)row * ldo + (size_t)(kvh * G + gt * 16 + hg) * d + e] = float_to_bf16(acc / l);
    }
  }
  if constexpr (LAST) {
    // The block's partial result for every head of the tile: the waves' results added in wave order, not divided by
    // the sum; to parts[row][head][block][d + 2] = o, maximum, sum.
    __syncthreads();
    const int stride = d + 2, nz = blk.ranges, z = blk.range;
    for (int idx = threadIdx.x; idx < tile_heads * d; idx += NW * 64) {
      const int hg = idx / d, e = idx % d;
      const float* src = meet + (size_t)hg * stride;
      float m = -INFINITY;
#pragma unroll
      for (int w = 0; w < NW; ++w) m = fmaxf(m, src[(size_t)w * tile_heads * stride + d]);
      float l = 0.f, acc = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float* ws = src + (size_t)w * tile_heads * stride;
        const float pm = ws[d];
        const float wgt = pm == -INFINITY ? 0.f : exp2_neg(pm - m);
        l += ws[d + 1] * wgt;
        acc = fmaf(ws[e], wgt, acc);
      }
      float* dst = parts + (((size_t)ri * H + (kvh * G + gt * 16 + hg)) * nz + z) * stride;
      st_coh(dst + e, acc);
      if (e == 0) {
        st_coh(dst + d, m);
        st_coh(dst + d + 1, l);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's stores have reached memory
    __syncthreads();
    int* counter = counters + (size_t)ri * blk.pairs + blk.pair;
    if (threadIdx.x == 0) {
      const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *is_last = before == nz - 1;
      if (*is_last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
    __syncthreads();
    if (!*is_last) return;
    // the last block of the pair: the blocks' results of every head, in block order (only blocks with a visible key)
    const int p_lo = (seen0 - base) / KW, p_hi = min((pos - base) / KW, n_parts - 1);
    const int z_lo = p_lo / NW, nzv = p_hi / NW - z_lo + 1;
    if (nzv <= LAST_DIRECT) {
      // few blocks: a thread asks for the maxima, sums and its element of all of them at once (one trip to memory
      // where the general way below makes two with a barrier between); the same additions in the same order
      for (int idx = threadIdx.x; idx < tile_heads * d; idx += NW * 64) {
        const int hg = idx / d, e = idx % d;
        const float* src = parts + (((size_t)ri * H + (kvh * G + gt * 16 + hg)) * nz + z_lo) * stride;
        float pm[LAST_DIRECT], pl[LAST_DIRECT], po[LAST_DIRECT];
#pragma unroll
        for (int zz = 0; zz < LAST_DIRECT; ++zz) {
          const float* sz = src + (size_t)min(zz, nzv - 1) * stride;
          pm[zz] = ld_coh(sz + d);
          pl[zz] = ld_coh(sz + d + 1);
          po[zz] = ld_coh(sz + e);
        }
        float m = -INFINITY;
#pragma unroll
        for (int zz = 0; zz < LAST_DIRECT; ++zz)
          if (zz < nzv) m = fmaxf(m, pm[zz]);
        float l = 0.f, acc = 0.f;
#pragma unroll
        for (int zz = 0; zz < LAST_DIRECT; ++zz)
          if (zz < nzv) {
            const float wgt = pm[zz] == -INFINITY ? 0.f : exp2_neg(pm[zz] - m);
            l += pl[zz] * wgt;
            acc = fmaf(po[zz], wgt, acc);
          }
        out[(size_t)row * ldo + (size_t)(kvh * G + gt * 16 + hg) * d + e] = float_to_bf16(acc / l);
      }
      return;
    }
    float* ml = meet;  // [heads of the tile][nzv][2]: maximum, sum (the waves' results are not needed any more)
    for (int idx = threadIdx.x; idx < tile_heads * nzv; idx += NW * 64) {
      const int hg = idx / nzv, zz = idx % nzv;
      const float* src = parts + (((size_t)ri * H + (kvh * G + gt * 16 + hg)) * nz + z_lo + zz) * stride;
      ml[idx * 2] = ld_coh(src + d);
      ml[idx * 2 + 1] = ld_coh(src + d + 1);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < tile_heads * d; idx += NW * 64) {
      const int hg = idx / d, e = idx % d;
      const float* src = parts + (((size_t)ri * H + (kvh * G + gt * 16 + hg)) * nz + z_lo) * stride + e;
      const float* mlh = ml + (size_t)hg * nzv * 2;
      float m = -INFINITY;
      for (int zz = 0; zz < nzv; ++zz) m = fmaxf(m, mlh[zz * 2]);
      float l = 0.f, acc = 0.f;
      for (int zz = 0; zz < nzv; ++zz) {
        const float pm = mlh[zz * 2];
        const float wgt = pm == -INFINITY ? 0.f : exp2_neg(pm - m);
        l += mlh[zz * 2 + 1] * wgt;
        acc = fmaf(ld_coh(src + (size_t)zz * stride), wgt, acc);
      }
      out[(size_t)row * ldo + (size_t)(kvh * G + gt * 16 + hg) * d + e] = float_to_bf16(acc / l);
    }
  }
}

}  // namespace attn_decode
