// attn_decode.h - the decode attention as per-wave device functions (attention.hip: one wave per (kv head, tile slot, sequence), the
// partials merged by a second launch).  Two other forms were built on these functions, measured and removed: one workgroup per (kv
// head, sequence) merging in LDS (round 4, profiles/r4_attn_wg_ab.txt) and the merge by the last-arriving waves of the same launch
// (round 5, profiles/r5_attn_fold_ab.txt: 16.1 us against 8.95 + 4.88 - five dependent round trips behind the last arriver).
#pragma once
#include <math.h>

#include "common.h"

namespace chatts {

constexpr int kMaxGroup = 8;
constexpr int kTile = 64;    // prefill kernel: keys per tile
constexpr int kDTile = 16;   // decode kernel: keys per wave-tile
constexpr int kMaxSlots = 64;    // decode: tile slots per kv head (one lane of the combine wave each)

struct AttnParams {
  const float* qkv;   // [T, (n_q + 2 n_kv) * 128]; q already rotated for attn_rows, raw for attn_decode
  float* kc;          // [n_kv, max_ctx, 128]
  float* vc;
  float* out;         // [T, n_q * 128]
  float* part_ml;     // [T, n_q, n_splits, 2]
  float* part_o;      // [T, n_q, n_splits, 128]
  const int32_t* pos0_dev;
  int pos0, t, n_q, n_kv, max_ctx, n_splits;
  // decode only
  const float* q_norm_w;
  const float* k_norm_w;
  const float* cos_tab;
  const float* sin_tab;
  float eps;
  size_t seq_stride;   // batched decode: floats between the caches of consecutive sequences (same layer)
  // block-paged cache (ChattsKvCache.block_table != NULL): kc / vc are the layer's pool [n_blocks, n_kv, 2^log_block, 128];
  // sequence b looks its blocks up in table + b * table_stride, seq_stride is not used
  const int32_t* table;
  int log_block, table_stride;
  uint16_t* out_hi;    // decode combine, optional: the output as bf16 hi / lo planes [T, n_q * 128] (the o_proj operand of the
  uint16_t* out_lo;    // weight-streaming kernel) instead of float32 `out`
  int out_tiled;       // prefill: so many rows of out_hi / out_lo in tiles (plane_at)
  int kv_round;        // experiment knob, see kv_round_f (0 = off)
  // prefill (bf16x3 kernel), optional: this sequence's K / V rows 0 .. kv_plane_keys-1 already split into bf16 hi / lo planes by
  // kv_planes_kernel (its layout is described there).  NULL: split while staging
  const uint16_t* kv_planes;
  int kv_plane_tiles;  // tiles per kv head
  // attn_prefill_planes_kernel's 1-D grid: query tiles per head and, when n_kv divides 8, the number of XCDs that share one kv head
  // (8 / n_kv; 0 = no XCD-aware order) - see the kernel
  int units, xcd_share;
  // decode: qkv points at the splits that the projection left (SplitSums), qkv_splits of them, floats qkv_plane apart; their sums times qkv_scale plus qkv_bias (either may be NULL)
  size_t qkv_plane;
  const float *qkv_scale, *qkv_bias;
  int qkv_splits;
};

// rotate one 128-wide head held as (a = x[lane], b = x[lane+64]) by the wave; optional RMSNorm first
__device__ __forceinline__ void norm_rope(float& a, float& b, const float* nw, float eps, float c, float s, int lane) {
  // every instantiation of the decode attention (stand-alone, persistent step) must produce the SAME bits here: no contraction
  // decisions left to the optimiser (seen: an unrelated statement after this call flipped one instantiation's a * c - b * s to an fma)
#pragma clang fp contract(off)
  if (nw) {
    const float ss = wave_sum(a * a + b * b);
    const float rstd = rsqrtf(ss / (float)kHeadDim + eps);
    a = nw[lane] * (a * rstd);
    b = nw[lane + 64] * (b * rstd);
  }
  const float oa = a * c - b * s, ob = b * c + a * s;
  a = oa;
  b = ob;
}

__device__ __forceinline__ float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// ---------------------------------------------------------------------------------------------------
// decode: grid (n_kv, n_slots), 64 threads.  Slot s of S (attn_slots) walks tiles s, s + S, ... of 16 keys.
//
// What bounds it: with few sequences a chain of latencies, with many the cache's bytes (8 KB a key of 8 kv heads) and, next to them, the vector pipe: five heads a row are 10 FMAs a float
// of K and V.  A tile was ~800 instructions, half of them softmax and weights that crossed lanes; a wave held two tiles in registers, one to work on and one under way.  Now a
// tile is ~480: K's registers take the next tile as soon as the scores are there, V's after the second product.
// Both launches in a graph over rotating caches, us before (with the merge as it is) / now: 16 sequences at 1204, 40 heads 36.9 / 30.8; 5 at 801, 32 heads 14.4 / 13.9; 8 at 800, 40 heads
// 20.3 / 17.9; one at 1800 13.8 / 11.6; groups of 8: 4 sequences at 1200 29.1 / 18.9.
// ---------------------------------------------------------------------------------------------------
constexpr float kNoKeys = -3.0e38f;      // a softmax's reference before its first key (finite: its distance to any reference is one, or -inf)
// halves: the lower 32 lanes get the sum of x over both halves, the upper 32 that of y; rows of 16 lanes: even rows the sum of x over a pair of rows, odd ones that of y
__device__ __forceinline__ float swap_add32(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap_add16(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One wave's work: kv head hk, tile slot `slot` of sequence `seq`, in two stages:
//   attn_decode_preload: everything that does not depend on this step's qkv - the position, the slot's first K tile, cos / sin;
//   attn_decode_finish : q prologue, new K / V row, scores, softmax, P.V, the partial.
// q_s [GMAX * 128], knew_s / vnew_s [128] are LDS scratch of the wave (16-byte aligned).  The partial of head g goes to part_o[(head_base + g0 + g) * NS + slot] / part_ml[..].
struct AttnTileRegs {       // what a wave keeps between the two stages: the slot's first K tile, cos / sin, the position
  f32x4 kv[8];
  float c, s;
  int pos;
};

// Register layout of a 16-key tile, K and V alike: lane = (kg = lane >> 3, c = lane & 7) holds dims c*4 + 32 i (i < 4) of key kg in r[i] and of key 8 + kg in r[4 + i]: one
// instruction = 8 key rows x 128 contiguous bytes (whole lines: a request of 16 rows x 64 bytes, the MFMA operand shape, streams at 4.1 TB/s on this part, whole lines at 6.2,
// profiles/r3_row_stream_probe.txt).  A key's score ends up in the 8 lanes that hold its V row, so nothing crosses lanes between the two products.
// A decode step reads every cache row exactly once: the tile loads are non-temporal like the weight stream (they do not displace the
// activations and partials the step re-reads from L2).  Measured A/B (-DCHATTS_KV_NT=0 builds the plain loads): config 5 6.51 -> 6.24 ms
// per step, config 4 162.4 -> 164.1 tok/s, headline 180.4 -> 181.7 tok/s.
#ifndef CHATTS_KV_NT
#define CHATTS_KV_NT 1
#endif
__device__ __forceinline__ f32x4 kv_stream_load(const float* p) {
#if CHATTS_KV_NT
  return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
#else
  return *reinterpret_cast<const f32x4*>(p);
#endif
}
__device__ __forceinline__ void attn_load_rows(const KvLayout& kvl, const float* cache, const int hk, const int tile, const int pos,
                                               const int lane, f32x4 (&r)[8]) {
  const int kg = lane >> 3, c = lane & 7;
  const int j0 = tile * kDTile;
  const int last = pos - j0;                              // clamped addresses (stay inside this tile: pos lies in it); masked below
  const unsigned a = (unsigned)((kg <= last ? kg : last) * kHeadDim + c * 4), b = (unsigned)((8 + kg <= last ? 8 + kg : last) * kHeadDim + c * 4);
  const float* rows = cache + kv_tile_off(kvl, hk, j0);   // the tile's first row: one table lookup per tile when the cache is paged
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = kv_stream_load(rows + a + i * 32);
#pragma unroll
  for (int i = 0; i < 4; ++i) r[4 + i] = kv_stream_load(rows + b + i * 32);
}

// Slots that a context of so many tiles uses: one for each tile as far as they go, else as few as do with the same number of tiles in the longest of them (a wave more costs its prologue
// and a row of the merge, a tile more in one of them 1.2 us for all: 3 sequences of 50 tiles, 40 heads, 42 slots of one or two tiles 13.3 us for both launches, 25 to 32 of two 13.0).
__device__ __forceinline__ int attn_slots(const int ntiles, const int n_splits) {
  if (ntiles <= n_splits) return ntiles;
  const unsigned longest = ((unsigned)ntiles + n_splits - 1) / (unsigned)n_splits;
  return (int)(((unsigned)ntiles + longest - 1) / longest);
}

// -> false: nothing to do for this slot (parked sequence, or the slot lies beyond the context)
__device__ __forceinline__ bool attn_decode_preload(const AttnParams& p, const int hk, const int slot, const int seq, const int lane,
                                                    AttnTileRegs& t) {
  const int pos = p.pos0_dev ? p.pos0_dev[seq] : p.pos0;     // batched decode: one position per sequence
  t.pos = pos;
  if (pos < 0) return false;                   // parked slot of a batched step: no cache write, no attention (its row is ignored)
  const int ntiles = pos / kDTile + 1;
  if (slot >= attn_slots(ntiles, p.n_splits)) return false;      // (the merge reads no others)
  const float* kcache = p.kc + (p.table ? 0 : (size_t)seq * p.seq_stride);
  const KvLayout kvl{p.table ? p.table + (size_t)seq * p.table_stride : nullptr, p.n_kv, p.max_ctx, p.log_block};
  // K of the first tile only depends on `pos`: issued before the q prologue so that the cache rows, q, cos / sin all travel in
  // the same memory round trip (or, preloaded, in an earlier one); V follows at the head of the second stage - it is not
  // needed before the softmax is done
  attn_load_rows(kvl, kcache, hk, slot, pos, lane, t.kv);
  t.c = p.cos_tab[(size_t)pos * 64 + lane];
  t.s = p.sin_tab[(size_t)pos * 64 + lane];
  return true;
}

// GMAX: query heads of the group this wave handles at most; it takes heads g0 .. g0 + gn - 1 of kv head hk's group (two waves share a group of 7 or 8).  Heads are independent of each
// other, so the split does not change a single operation of any head.  The wave with g0 == 0 stores the new K / V row.
// EXACT: the group IS GMAX heads - `g < gn` is decided by the compiler and the tile body is one straight-line block (the
// run-time form compiled to ~400 basic blocks, every head's every step behind a scalar branch, no load / FMA interleaving across them).
// SPLITS: up to so many splits of qkv are summed here (splitk_epilogue_v4_kernel's order: the same bits), 0: qkv is whole
// (a wave reads so many times 3.5 KB instead of 3.5, all of them requested at once, and a launch of 2.5 us that only sums falls away: a step of ChatTS-14B, fp8, 16 sequences at 1204, four
// splits: 5300 -> 5170 us.)
template <int GMAX, bool EXACT, int SPLITS>
__device__ __forceinline__ void attn_decode_finish(const AttnParams& p, const int hk, const int slot, const int seq, const int lane,
                                                   AttnTileRegs& t, float* q_s, float* knew_s, float* vnew_s, const int g0, const int gn_rt,
                                                   float* part_o, float* part_ml, const size_t head_base) {
  const int gn = EXACT ? GMAX : gn_rt;
  const int G = EXACT ? GMAX : p.n_q / p.n_kv;
  const int pos = t.pos;
  const int ntiles = pos / kDTile + 1, NS = p.n_splits, walk = attn_slots(ntiles, NS);
  const int qkv_n = (p.n_q + 2 * p.n_kv) * kHeadDim;
  const float* qkv = p.qkv + (size_t)seq * qkv_n;
  // a head of 128 as (x[lane], x[lane + 64]): what is requested for it, and its values once that is there
  struct Head { float a[SPLITS ? SPLITS : 1], b[SPLITS ? SPLITS : 1], fa, fb, ba, bb; };
  auto request = [&](Head& h, const int col) __attribute__((always_inline)) {
    const float* at = qkv + col + lane;
    if constexpr (SPLITS == 0) {
      h.a[0] = at[0];
      h.b[0] = at[64];
    } else {
#pragma unroll
      for (int i = 0; i < SPLITS; ++i) {
        const float* split = at + (i < p.qkv_splits ? i : p.qkv_splits - 1) * p.qkv_plane;
        h.a[i] = split[0];
        h.b[i] = split[64];
      }
      h.fa = h.fb = 1.f;
      h.ba = h.bb = 0.f;
      if (p.qkv_scale) { h.fa = p.qkv_scale[col + lane]; h.fb = p.qkv_scale[col + lane + 64]; }
      if (p.qkv_bias) { h.ba = p.qkv_bias[col + lane]; h.bb = p.qkv_bias[col + lane + 64]; }
    }
  };
  auto value = [&](const Head& h, float& a, float& b) __attribute__((always_inline)) {
    if constexpr (SPLITS == 0) {
      a = h.a[0];
      b = h.b[0];
    } else {
      a = b = 0.f;
#pragma unroll
      for (int i = 0; i < SPLITS; ++i)
        if (i < p.qkv_splits) { a += h.a[i]; b += h.b[i]; }
      a *= h.fa; b *= h.fb;
      if (p.qkv_bias) { a += h.ba; b += h.bb; }
    }
  };
  float* kcache = p.kc + (p.table ? 0 : (size_t)seq * p.seq_stride);
  float* vcache = p.vc + (p.table ? 0 : (size_t)seq * p.seq_stride);
  const KvLayout kvl{p.table ? p.table + (size_t)seq * p.table_stride : nullptr, p.n_kv, p.max_ctx, p.log_block};
  const bool owner = (ntiles - 1) % walk == slot;
  const float scale = 0.08838834764831845f * 1.4426950408889634f;    // 128^-1/2 * log2(e): the softmax runs on v_exp_f32 (exp2)
  const int kg = lane >> 3, kc = lane & 7;      // see attn_load_rows
  f32x4 (&kv)[8] = t.kv;
  f32x4 vv[8];
  attn_load_rows(kvl, vcache, hk, slot, pos, lane, vv);

  {
    const float c = t.c, s = t.s;
    Head q[GMAX];
#pragma unroll
    for (int g = 0; g < GMAX; ++g)
      if (g < gn) request(q[g], (hk * G + g0 + g) * kHeadDim);
#pragma unroll
    for (int g = 0; g < GMAX; ++g) {
      if (g < gn) {
        float a, b;
        value(q[g], a, b);
        norm_rope(a, b, p.q_norm_w, p.eps, c, s, lane);
        q_s[g * kHeadDim + lane] = a;
        q_s[g * kHeadDim + lane + 64] = b;
      }
    }
    if (owner) {                                // the new K/V row: to the cache and to LDS
      Head kh, vh;
      request(kh, (p.n_q + hk) * kHeadDim);
      request(vh, (p.n_q + p.n_kv + hk) * kHeadDim);
      float a, b;
      value(kh, a, b);
      norm_rope(a, b, p.k_norm_w, p.eps, c, s, lane);
      a = kv_round_f(a, p.kv_round); b = kv_round_f(b, p.kv_round);
      knew_s[lane] = a;
      knew_s[lane + 64] = b;
      const size_t noff = kv_tile_off(kvl, hk, pos);      // row of the new token
      float* kd = kcache + noff;
      if (g0 == 0) { kd[lane] = a; kd[lane + 64] = b; }
      float va, vb;
      value(vh, va, vb);
      va = kv_round_f(va, p.kv_round);
      vb = kv_round_f(vb, p.kv_round);
      vnew_s[lane] = va;
      vnew_s[lane + 64] = vb;
      float* vd = vcache + noff;
      if (g0 == 0) { vd[lane] = va; vd[lane + 64] = vb; }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // single wave: orders the LDS writes above (in-order LDS, no barrier needed)

  // Every 8 lanes (kg) run a softmax of their own over the keys that they hold, and meet the other groups behind the last tile: a tile has no reduction over the wave.  A group's
  // reference m moves only when a score lies more than kSlack (a factor of 256) above it, so the sums are seldom rescaled; what is exponentiated stays below 2^8 either way.
  constexpr float kSlack = 8.f;
  float m_run[GMAX], l_run[GMAX];
  f32x4 acc[GMAX][4];                           // this lane's 16 dims, summed over its group's keys
#pragma unroll
  for (int g = 0; g < GMAX; ++g) {
    m_run[g] = kNoKeys; l_run[g] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[g][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  // the row just produced is not in the cache for this wave yet; rows behind it hold anything
  auto new_row = [&](const int tile, f32x4 (&r)[8], const float* row_s) __attribute__((always_inline)) {
    if (tile != ntiles - 1) return;
    const int ja = tile * kDTile + kg;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(row_s + kc * 4 + i * 32);
      if (ja >= pos) r[i] = v;
      if (ja + 8 >= pos) r[4 + i] = v;
    }
  };
  for (int tile = slot; tile < ntiles; tile += walk) {
    const int ja = tile * kDTile + kg, jb = ja + 8, next = tile + walk;
    if (owner) new_row(tile, kv, knew_s);
    float pa[GMAX], pb[GMAX];
#pragma unroll
    for (int g = 0; g < GMAX; ++g) { pa[g] = 0.f; pb[g] = 0.f; }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int g = 0; g < GMAX; ++g) {
        if (g < gn) {
          const f32x4 qv = *reinterpret_cast<const f32x4*>(q_s + g * kHeadDim + kc * 4 + i * 32);      // shared by both keys
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            pa[g] = fmaf(kv[i][e], qv[e], pa[g]);
            pb[g] = fmaf(kv[4 + i][e], qv[e], pb[g]);
          }
        }
      }
      // EXACT: keep the q fragments of one 32-dim slice live at a time (unfenced, the scheduler hoists all GMAX x 4 LDS reads of the
      // tile to its top and the kernel no longer fits the 256 registers of two waves per SIMD)
      if constexpr (EXACT) __builtin_amdgcn_sched_barrier(0);
    }
    // (the compiler sinks sums towards their uses, past the loads that follow: K and V would then need two sets of registers)
#pragma unroll
    for (int g = 0; g < GMAX; ++g) asm volatile("" : "+v"(pa[g]), "+v"(pb[g]));
    if (next < ntiles) attn_load_rows(kvl, kcache, hk, next, pos, lane, kv);      // (K's registers are free, V's behind the second product)
    float above = -INFINITY;
#pragma unroll
    for (int g = 0; g < GMAX; ++g) {
      if (g < gn) {
        float sa = pa[g], sb = pb[g];
        sa += lane_xor1(sa); sb += lane_xor1(sb);
        sa += lane_xor2(sa); sb += lane_xor2(sb);
        sa += half_mirror(sa); sb += half_mirror(sb);      // all 8 lanes of a key pair now hold both scores (DPP, no LDS round trip)
        pa[g] = ja <= pos ? sa * scale : -INFINITY;
        pb[g] = jb <= pos ? sb * scale : -INFINITY;
        above = fmaxf(above, fmaxf(pa[g], pb[g]) - m_run[g]);
      }
    }
    if (__builtin_amdgcn_ballot_w64(above > kSlack)) {
#pragma unroll
      for (int g = 0; g < GMAX; ++g) {
        if (g < gn) {
          const float m_new = fmaxf(m_run[g], fmaxf(pa[g], pb[g]));
          const float alpha = __builtin_amdgcn_exp2f(m_run[g] - m_new);
          m_run[g] = m_new;
          l_run[g] *= alpha;
          if (tile != slot) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[g][i][e] *= alpha;
          }
        }
      }
    }
#pragma unroll
    for (int g = 0; g < GMAX; ++g) {
      if (g < gn) {
        pa[g] = __builtin_amdgcn_exp2f(pa[g] - m_run[g]);
        pb[g] = __builtin_amdgcn_exp2f(pb[g] - m_run[g]);
        l_run[g] += pa[g] + pb[g];
      }
    }
    if (owner) new_row(tile, vv, vnew_s);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int g = 0; g < GMAX; ++g) {
        if (g < gn) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[g][i][e] = fmaf(pb[g], vv[4 + i][e], fmaf(pa[g], vv[i][e], acc[g][i][e]));
        }
      }
      if constexpr (EXACT) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int g = 0; g < GMAX; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(acc[g][i]));
    if (next < ntiles) attn_load_rows(kvl, vcache, hk, next, pos, lane, vv);
  }
  f32x4 o[GMAX];
  float M[GMAX], l[GMAX];
#pragma unroll
  for (int g = 0; g < GMAX; ++g) {
    if (g < gn) {
      M[g] = rows4_max(fmaxf(m_run[g], row_ror8(m_run[g])));
      const float f = __builtin_amdgcn_exp2f(m_run[g] - M[g]);      // (0 for a group without keys)
      const float lf = l_run[g] * f;
      l[g] = rows4_sum(lf + row_ror8(lf));
#pragma unroll
      for (int e = 0; e < 4; ++e) {             // the 8 groups' sums; row r of 16 lanes ends up with dims 32 r ..
        const float x = swap_add32(acc[g][0][e] * f, acc[g][2][e] * f), y = swap_add32(acc[g][1][e] * f, acc[g][3][e] * f);
        const float z = swap_add16(x, y);
        o[g][e] = z + row_ror8(z);
      }
    }
  }
  const size_t p0 = (head_base + g0) * NS + slot;
  if (!(lane & 8)) {
#pragma unroll
    for (int g = 0; g < GMAX; ++g)
      if (g < gn) *reinterpret_cast<f32x4*>(part_o + (p0 + (size_t)g * NS) * kHeadDim + (lane >> 4) * 32 + kc * 4) = o[g];
  }
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < GMAX; ++g)
      if (g < gn) *reinterpret_cast<u32x2*>(part_ml + (p0 + (size_t)g * NS) * 2) = (u32x2){__float_as_uint(M[g] * 0.6931471805599453f), __float_as_uint(l[g])};      // (m back to nats for the combine)
  }
}


// GMAX >= the heads of this wave: the per-head registers are sized by it
template <int GMAX, bool EXACT, int SPLITS>
__device__ __forceinline__ void attn_decode_wave(const AttnParams& p, const int hk, const int slot, const int seq, const int lane,
                                                 float* q_s, float* knew_s, float* vnew_s, const int g0, const int gn, float* part_o, float* part_ml,
                                                 const size_t head_base) {
  AttnTileRegs t;
  if (!attn_decode_preload(p, hk, slot, seq, lane, t)) return;
  attn_decode_finish<GMAX, EXACT, SPLITS>(p, hk, slot, seq, lane, t, q_s, knew_s, vnew_s, g0, gn, part_o, part_ml, head_base);
}

// out[h] = sum_s e^{m_s - M} o_s / sum_s e^{m_s - M} l_s over the slots that saw keys (<= CAP of them).
// One wave's half of a head: d = half * 64 + lane (two waves per head).  The partials of head hq are part_o / part_ml rows base .. base + n_splits - 1.
// This launch is a chain of latencies and nothing else.  (m, l) and all rows of this lane's dim are requested before the position is there: nothing that is loaded
// depends on it, only what is summed does (rows of slots that saw no keys hold anything and stay out).  One buffer with immediate offsets: an address for each row was
// ~500 scalar instructions ahead of the first load.  The weights are read from their lanes, not through LDS.  CAP: the least of 16, 32, 64 that holds n_splits.
template <int CAP>
__device__ __forceinline__ void attn_combine_wave(const AttnParams& p, const int hq, const int seq, const int d, const int lane,
                                                  const float* part_o, const float* part_ml, const size_t base) {
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc((void*)(part_o + base * kHeadDim), 0, p.n_splits * kHeadDim * (int)sizeof(float), 0x00020000);
  float o[CAP];
#pragma unroll
  for (int u = 0; u < CAP; ++u) o[u] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, d * (int)sizeof(float) + u * 512, 0, 0));      // (0 behind the last slot)
  float m = -INFINITY, l = 0.f;
  if (lane < p.n_splits) { m = part_ml[(base + lane) * 2]; l = part_ml[(base + lane) * 2 + 1]; }
  const int pos = p.pos0_dev ? p.pos0_dev[seq] : p.pos0;
  const int ntiles = pos < 0 ? 0 : pos / kDTile + 1;         // parked slot: no partials exist, the row is written as zeros
  const int ns = attn_slots(ntiles, p.n_splits);
  const float M = wave_max(lane < ns ? m : -INFINITY);
  const float w = lane < ns ? expf(m - M) : 0.f;
  const float den = wave_sum(lane < ns ? w * l : 0.f);
  float num = 0.f;
#pragma unroll
  for (int u0 = 0; u0 < CAP; u0 += 8) {
    if (u0 < ns) {
#pragma unroll
      for (int u = u0; u < u0 + 8; ++u) num = fmaf(readlane_f(w, u), u < ns ? o[u] : 0.f, num);      // (slots in ascending order)
    }
  }
  const size_t oi = ((size_t)seq * p.n_q + hq) * kHeadDim + d;
  const float v = ns > 0 ? num / den : 0.f;
  if (p.out_hi) {
    const __bf16 h = (__bf16)v;
    p.out_hi[oi] = __builtin_bit_cast(uint16_t, h);
    p.out_lo[oi] = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)h));
  } else {
    p.out[oi] = v;
  }
}

}  // namespace chatts
