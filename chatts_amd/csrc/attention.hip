// attention.hip - causal grouped-query attention over the float32 KV cache (head_dim 128).
// Math per transformers eager_attention_forward (oracle/qwen_decoder.py): scores = q.k^T * d^-1/2,
// float32 softmax, out = P.V; GQA: the n_q/n_kv query heads of a group share one K/V head (repeat_kv).
//
// Kernels:
//  * attn_decode_kernel (T = 1, the per-token path): ONE WAVE per (kv head, 16-key tile).  A wave has no
//    barriers to wait for, issues all of its K (8 x 16 B) and V (16 x 8 B) loads at once and finishes in about
//    one memory round trip; hundreds of such waves spread the cache read over all CUs.  It also fuses what
//    used to be a separate launch: per-head q/k RMSNorm (Qwen3), RoPE of q and of the new k, and the write of
//    the new K/V row into the cache (done by the single wave whose tile contains `pos`, which then uses the row
//    from LDS).  Softmax statistics are wave shuffles; P is broadcast lane->wave with v_readlane.
//    Each wave emits an (m, l, o[G][128]) partial; attn_decode_combine_kernel merges the partials of a head.
//  * attn_rows_kernel (short prefill chunks, T < 16, and the last-row path): one workgroup per (kv head, query row), 64-key
//    tiles, online softmax, float32 VALU.  Longer chunks run the flash kernels further down: attn_prefill_bf16x3_kernel (bf16
//    matrix pipe on hi / lo planes, the default) and attn_prefill_mfma_kernel (exact-f32 MFMA).
// The KV cache is float32 on purpose: the parity target is the float32 reference path and the cache
// is ~1% of decode traffic at the benchmark context.
#include <math.h>

#include "common.h"

namespace chatts {

}  // namespace chatts
#include "attn_decode.h"
#include "gemm_common.h"
namespace chatts {

// ---------------------------------------------------------------------------------------------------
// decode: grid (n_kv, n_splits, sequences), 64 threads; TWO: (n_kv, 2 n_splits, sequences).  Slot s of the S that a context uses (attn_slots, at most n_splits) walks tiles s, s + S, ...
// of 16 keys; the others leave.
// ---------------------------------------------------------------------------------------------------
// TWO: groups of 7 and 8 heads, whose sums do not fit the registers of two waves per SIMD: two waves a slot, four heads and the rest, next to each other on one XCD (a row of the
// cache comes from memory once).  One wave per SIMD with all heads was 1.1 .. 1.4 times slower from 12 sequences on, spilling 10 registers 1.1 .. 1.3 times nearly everywhere.
template <int GMAX, bool EXACT, bool TWO = false, int SPLITS = 0>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void attn_decode_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) float q_s[GMAX * kHeadDim];
  __shared__ __attribute__((aligned(16))) float knew_s[kHeadDim];
  __shared__ __attribute__((aligned(16))) float vnew_s[kHeadDim];
  const int group = EXACT ? GMAX : p.n_q / p.n_kv, g0 = TWO ? ((int)blockIdx.y & 1) * GMAX : 0;
  attn_decode_wave<GMAX, EXACT, SPLITS>(p, blockIdx.x, TWO ? blockIdx.y >> 1 : blockIdx.y, blockIdx.z, threadIdx.x, q_s, knew_s, vnew_s, g0, group - g0 < GMAX ? group - g0 : GMAX, p.part_o,
                                p.part_ml, (size_t)blockIdx.z * p.n_q + blockIdx.x * group);
}

// out[h] = sum_s e^{m_s - M} o_s / sum_s e^{m_s - M} l_s over the slots that saw keys (<= 64 slots): attn_combine_wave
// (attn_decode.h), one workgroup (2 waves) per head.
template <int CAP>
__global__ __launch_bounds__(128) void attn_decode_combine_kernel(AttnParams p) {
  attn_combine_wave<CAP>(p, blockIdx.x, blockIdx.y, threadIdx.x, threadIdx.x & 63, p.part_o, p.part_ml,
                    ((size_t)blockIdx.y * p.n_q + blockIdx.x) * p.n_splits);
}

// ---------------------------------------------------------------------------------------------------
// prefill: grid (n_kv, T, n_splits), 256 threads, 64-key tiles.
//   phase 1  scores: 4 lanes per key (32 dims each), xor-shuffle reduce
//   phase 2  one wave per head: tile max / rescale factor / p = exp(s - m) written back to LDS
//   phase 3  P.V: thread = (dim, key half), V rows read fully coalesced, 8 loads in flight per thread
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void attn_rows_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) float q_s[kMaxGroup * kHeadDim];
  __shared__ float s_s[kMaxGroup * kTile];
  __shared__ float alpha_s[kMaxGroup];
  __shared__ float o_s[kMaxGroup * kHeadDim];

  const int hk = blockIdx.x, row = blockIdx.y, split = blockIdx.z;
  const int G = p.n_q / p.n_kv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int pos = (p.pos0_dev ? *p.pos0_dev : p.pos0) + row;
  const int heads = p.n_q + 2 * p.n_kv;
  const float scale = 0.08838834764831845f;
  const int ntiles = pos / kTile + 1;

  for (int i = tid; i < G * kHeadDim; i += 256)
    q_s[i] = p.qkv[((size_t)row * heads + hk * G) * kHeadDim + i];
  __syncthreads();

  const KvLayout kvl{p.table, p.n_kv, p.max_ctx, p.log_block};
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};   // heads wave, wave + 4
  float acc[kMaxGroup];
#pragma unroll
  for (int g = 0; g < kMaxGroup; ++g) acc[g] = 0.f;
  const int key_l = tid >> 2, quarter = tid & 3;
  const int d_o = tid & 127, half = tid >> 7;

  for (int tile = split; tile < ntiles; tile += p.n_splits) {
    const int j0 = tile * kTile;
    const size_t toff = kv_tile_off(kvl, hk, j0);     // first row of the tile (one block-table lookup when paged)
    {
      const int j = j0 + key_l;
      const int jc = j <= pos ? j : pos;
      const float* kr = p.kc + toff + (size_t)(jc - j0) * kHeadDim + quarter * 4;
      f32x4 kv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) kv[i] = *reinterpret_cast<const f32x4*>(kr + i * 16);
      float dot[kMaxGroup];
#pragma unroll
      for (int g = 0; g < kMaxGroup; ++g) dot[g] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int g = 0; g < kMaxGroup; ++g) {
          if (g < G) {
            const f32x4 qv = *reinterpret_cast<const f32x4*>(q_s + g * kHeadDim + quarter * 4 + i * 16);
            dot[g] = fmaf(kv[i].x, qv.x, dot[g]);
            dot[g] = fmaf(kv[i].y, qv.y, dot[g]);
            dot[g] = fmaf(kv[i].z, qv.z, dot[g]);
            dot[g] = fmaf(kv[i].w, qv.w, dot[g]);
          }
        }
      }
#pragma unroll
      for (int g = 0; g < kMaxGroup; ++g) {
        if (g < G) {
          float v = dot[g];
          v += lane_xor1(v);
          v += lane_xor2(v);
          if (quarter == 0) s_s[g * kTile + key_l] = j <= pos ? v * scale : -INFINITY;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      const int g = wave + gi * 4;
      if (g < G) {
        const float s = s_s[g * kTile + lane];
        const float m_new = fmaxf(m_run[gi], wave_max(s));
        const float pr = expf(s - m_new);
        const float a = expf(m_run[gi] - m_new);
        l_run[gi] = l_run[gi] * a + wave_sum(pr);
        m_run[gi] = m_new;
        s_s[g * kTile + lane] = pr;
        if (lane == 0) alpha_s[g] = a;
      }
    }
    __syncthreads();
    {
#pragma unroll
      for (int g = 0; g < kMaxGroup; ++g)
        if (g < G) acc[g] *= alpha_s[g];
      const int jb = j0 + half * 32;
#pragma unroll
      for (int b8 = 0; b8 < 32; b8 += 8) {
        float vv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int j = jb + b8 + u;
          vv[u] = p.vc[toff + (size_t)((j <= pos ? j : pos) - j0) * kHeadDim + d_o];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
#pragma unroll
          for (int g = 0; g < kMaxGroup; ++g)
            if (g < G) acc[g] = fmaf(s_s[g * kTile + half * 32 + b8 + u], vv[u], acc[g]);   // p = 0 for masked keys
        }
      }
    }
    __syncthreads();
  }

  if (half == 1) {
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
      if (g < G) o_s[g * kHeadDim + d_o] = acc[g];
  }
  if (lane == 0) {
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      const int g = wave + gi * 4;
      if (g < G) { s_s[g * 2] = m_run[gi]; s_s[g * 2 + 1] = l_run[gi]; }
    }
  }
  __syncthreads();
  if (half == 0) {
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g) {
      if (g < G) {
        const float o = acc[g] + o_s[g * kHeadDim + d_o];
        const int hq = hk * G + g;
        if (p.n_splits == 1) {
          p.out[((size_t)row * p.n_q + hq) * kHeadDim + d_o] = o / s_s[g * 2 + 1];
        } else {
          const size_t pi = ((size_t)row * p.n_q + hq) * p.n_splits + split;
          p.part_o[pi * kHeadDim + d_o] = o;
          if (d_o == 0) { p.part_ml[pi * 2] = s_s[g * 2]; p.part_ml[pi * 2 + 1] = s_s[g * 2 + 1]; }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// prefill, flash style on the exact-f32 matrix cores (v_mfma_f32_16x16x4_f32: f32 in, f32 accumulate, bitwise an
// fmaf chain - the parity target is the float32 reference, and attention is ~3 % of prefill FLOPs, so the f32 MFMA
// rate (155 TF) is enough).  grid (ceil(T/64), n_q), 256 threads: wave w owns query rows q0+16w .. +15 of ONE q head.
//   Q fragment  A[i = lane&15][K-slot group lane>>4 = head dims 32*(lane>>4) ..+31]: 32 floats per lane, loaded once
//   K tile      [KT][136] f32 in LDS: B fragments are ds_read_b128 (4 MFMAs per read), conflict-free with the rotation kq & 1
//   S = Q.K^T   KT/16 accumulators in C layout (col = lane&15 = key, row = 4*(lane>>4) + reg)
//   softmax     online, per C-layout row: 16-lane xor shuffles for max and sum
//   P           C layout -> wave-private LDS [16][KT+2] -> A layout (row = lane&15, k = lane>>4 + 4j)
//   O += P.V    V tile [KT][132] f32 in LDS, 8 accumulators with permuted columns (lane n, acc db -> head dim 8n + db)
// Heaviest query tiles (most key tiles under the causal mask) are scheduled first (pairing heavy + light tiles in one
// workgroup was measured: slower, the chip then holds one wave per SIMD and nothing hides the per-tile overheads).
// ---------------------------------------------------------------------------------------------------
template <int KT>
__global__ __launch_bounds__(256, 3) void attn_prefill_mfma_kernel(AttnParams p) {
  constexpr int KS = 136, VS = 132, PS = KT + 2, NB = KT / 16;
  __shared__ __attribute__((aligned(16))) float v_s[KT * VS];
  __shared__ __attribute__((aligned(16))) float k_s[KT * KS];
  __shared__ float p_all[4 * 16 * PS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hq = blockIdx.y;
  const int G = p.n_q / p.n_kv, hk = hq / G;
  const int heads = p.n_q + 2 * p.n_kv;
  const int T = p.t, pos0 = p.pos0_dev ? *p.pos0_dev : p.pos0;
  const int qt = gridDim.x - 1 - blockIdx.x;                // heaviest query tiles (most key tiles) first
  const int q0 = qt * 64;
  const int arow = lane & 15, kq = lane >> 4;              // A/B fragment coordinates
  const int ccol = lane & 15, crow0 = (lane >> 4) * 4;     // C layout
  const float scale2 = 0.08838834764831845f * 1.4426950408889634f;   // d^-1/2 * log2(e): the softmax runs on exp2
  float* p_s = p_all + wave * 16 * PS;

  float qreg[32];
  {
    int qrow = q0 + wave * 16 + arow;
    if (qrow > T - 1) qrow = T - 1;                         // padded rows compute garbage that is never stored
    // K-slot assignment: the MFMA's K index is free as long as both operands agree, so lane group kq takes head dims
    // kq*32 .. kq*32+31 (contiguous: the K fragments below are ds_read_b128, four MFMAs per read), visiting its eight
    // 4-float chunks rotated by kq & 1 - the rotation that makes the b128 reads of the [KT][136] tile conflict-free.
    const float* qp = p.qkv + ((size_t)qrow * heads + hq) * kHeadDim + kq * 32;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x4 qv = *reinterpret_cast<const f32x4*>(qp + 4 * ((i + (kq & 1)) & 7));
      qreg[4 * i] = qv.x; qreg[4 * i + 1] = qv.y; qreg[4 * i + 2] = qv.z; qreg[4 * i + 3] = qv.w;
    }
  }
  int qpos[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) qpos[r] = pos0 + q0 + wave * 16 + crow0 + r;
  float m_run[4], l_run[4];
  f32x4 o_acc[8];
#pragma unroll
  for (int r = 0; r < 4; ++r) { m_run[r] = -INFINITY; l_run[r] = 0.f; }
#pragma unroll
  for (int db = 0; db < 8; ++db) o_acc[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int last_q = q0 + 63 < T - 1 ? q0 + 63 : T - 1;
  const int kmax = pos0 + last_q;                           // last key any row of this workgroup may see
  const int nkt = kmax / KT + 1;
  const KvLayout kvl{p.table, p.n_kv, p.max_ctx, p.log_block};

  // K/V tiles go global -> registers -> LDS; the loads of tile kt+1 are issued BEFORE the MFMAs of tile kt, so their L2
  // latency hides under the tile's 128 MFMAs per wave instead of sitting between two barriers.
  constexpr int SLOTS = KT * 32 / 256;                      // float4 slots per thread and operand
  f32x4 kreg[SLOTS], vreg[SLOTS];
  auto load_tile = [&](int kt) {
    const size_t toff = kv_tile_off(kvl, hk, kt * KT);      // first row of the tile (one block-table lookup when paged)
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int idx = tid + i * 256, key = idx >> 5, c4 = idx & 31;
      const int kr = kt * KT + key <= kmax ? key : kmax - kt * KT;    // clamped row inside the tile; masked by key index below
      kreg[i] = *reinterpret_cast<const f32x4*>(p.kc + toff + (size_t)kr * kHeadDim + c4 * 4);
      vreg[i] = *reinterpret_cast<const f32x4*>(p.vc + toff + (size_t)kr * kHeadDim + c4 * 4);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int idx = tid + i * 256, key = idx >> 5, c4 = idx & 31;
      *reinterpret_cast<f32x4*>(k_s + key * KS + c4 * 4) = kreg[i];
      *reinterpret_cast<f32x4*>(v_s + key * VS + c4 * 4) = vreg[i];
    }
  };
  // Key split (flash-decoding style): workgroup z takes key tiles z, z + NS, ...  T/16 x heads waves is all the parallelism one
  // sequence has (~2 waves per SIMD at T = 798, and the causal mask makes them unequal); splitting the keys doubles it.
  const int NS = p.n_splits, split = blockIdx.z;
  if (split < nkt) load_tile(split);
  for (int kt = split; kt < nkt; kt += NS) {
    const int k0 = kt * KT;
    __syncthreads();                                        // the previous tile has been consumed by every wave
    store_tile();
    __syncthreads();
    if (kt + NS < nkt) load_tile(kt + NS);

    f32x4 s_acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) s_acc[nb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f32x4 kf[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        kf[nb] = *reinterpret_cast<const f32x4*>(k_s + (nb * 16 + arow) * KS + kq * 32 + 4 * ((i + (kq & 1)) & 7));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          s_acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(qreg[4 * i + e], kf[nb][e], s_acc[nb], 0, 0, 0);
    }
    // Online softmax in the log2 domain (scores are pre-scaled by d^-1/2 * log2 e, so every exponential is one v_exp_f32),
    // written stage by stage over the four rows a lane holds: the DPP reductions are dependent chains with wait states,
    // and four independent chains in flight are what hides them (measured with s_memtime: this block was 3.5k cycles per
    // tile as a per-row loop with expf, against 2k cycles for the 64 MFMAs of Q.K^T).
    float mx[4], ps[4], alpha[4], m_ref[4];
    const bool diag = k0 + KT - 1 > pos0 + q0 + wave * 16;  // wave-uniform: only such a tile holds keys some row of this wave cannot see
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mx[r] = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        float sc = s_acc[nb][r] * scale2;
        if (diag && k0 + nb * 16 + ccol > qpos[r]) sc = -INFINITY;  // causal mask
        s_acc[nb][r] = sc;
        mx[r] = fmaxf(mx[r], sc);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], lane_xor1(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], lane_xor2(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], row_ror4(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], row_ror8(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float m_new = fmaxf(m_run[r], mx[r]);
      // a key split other than 0 may start on a tile this row cannot see at all: keep m = -inf, contribute nothing
      m_ref[r] = m_new == -INFINITY ? 0.f : m_new;
      alpha[r] = __builtin_amdgcn_exp2f(m_run[r] - m_ref[r]);
      m_run[r] = m_new;
      ps[r] = 0.f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float e = __builtin_amdgcn_exp2f(s_acc[nb][r] - m_ref[r]);
        s_acc[nb][r] = e;
        ps[r] += e;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += lane_xor1(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += lane_xor2(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += row_ror4(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += row_ror8(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      l_run[r] = l_run[r] * alpha[r] + ps[r];
#pragma unroll
      for (int db = 0; db < 8; ++db) o_acc[db][r] *= alpha[r];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) p_s[(crow0 + r) * PS + nb * 16 + ccol] = s_acc[nb][r];
    }
    __builtin_amdgcn_wave_barrier();                        // P is wave private: LDS ops of one wave stay in order
    // O += P.V with the output columns permuted: accumulator db of lane n holds head dim n*8 + db, so one key row gives a
    // lane its eight V values as two ds_read_b128 (conflict-free for the [KT][132] tile) and the final store is 32 B per lane
#pragma unroll
    for (int j = 0; j < KT / 4; ++j) {                      // unrolled: the reads of step j+1 are issued under the MFMAs of step j
      const float pa = p_s[arow * PS + kq + 4 * j];
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(v_s + (kq + 4 * j) * VS + arow * 8);
      const f32x4 v1 = *reinterpret_cast<const f32x4*>(v_s + (kq + 4 * j) * VS + arow * 8 + 4);
#pragma unroll
      for (int db = 0; db < 4; ++db) o_acc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v0[db], o_acc[db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < 4; ++db) o_acc[4 + db] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, v1[db], o_acc[4 + db], 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int qrow = q0 + wave * 16 + crow0 + r;
    if (qrow < T && NS > 1) {                               // partial (unnormalised) result of this key split
      const size_t pi = ((size_t)qrow * p.n_q + hq) * NS + split;
      float* dst = p.part_o + pi * kHeadDim + ccol * 8;
      *reinterpret_cast<f32x4*>(dst) = (f32x4){o_acc[0][r], o_acc[1][r], o_acc[2][r], o_acc[3][r]};
      *reinterpret_cast<f32x4*>(dst + 4) = (f32x4){o_acc[4][r], o_acc[5][r], o_acc[6][r], o_acc[7][r]};
      if (ccol == 0) { p.part_ml[pi * 2] = m_run[r] * 0.6931471805599453f; p.part_ml[pi * 2 + 1] = l_run[r]; }   // m back to nats
    } else if (qrow < T) {
      const float inv = 1.0f / l_run[r];
      const size_t oi = ((size_t)qrow * p.n_q + hq) * kHeadDim + ccol * 8;
      if (p.out_hi) {
        typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
        bf16x8v hv, lv;
#pragma unroll
        for (int db = 0; db < 8; ++db) {
#pragma clang fp contract(off)   // lo = split of the ROUNDED product, as chatts_split_bf16x2 of the float32 output would give
          const float v = o_acc[db][r] * inv;
          const __bf16 h = (__bf16)v;
          hv[db] = h;
          lv[db] = (__bf16)(v - (float)h);
        }
        const size_t at = plane_at(qrow, hq * kHeadDim + ccol * 8, p.n_q * kHeadDim, p.out_tiled);
        *reinterpret_cast<bf16x8v*>(p.out_hi + at) = hv;
        *reinterpret_cast<bf16x8v*>(p.out_lo + at) = lv;
      } else {
        float* dst = p.out + oi;
        *reinterpret_cast<f32x4*>(dst) = (f32x4){o_acc[0][r] * inv, o_acc[1][r] * inv, o_acc[2][r] * inv, o_acc[3][r] * inv};
        *reinterpret_cast<f32x4*>(dst + 4) = (f32x4){o_acc[4][r] * inv, o_acc[5][r] * inv, o_acc[6][r] * inv, o_acc[7][r] * inv};
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// prefill, bf16x3 form: the same flash loop as attn_prefill_mfma_kernel, but Q.K^T and P.V run on the bf16 matrix pipe
// (v_mfma_f32_16x16x32_bf16, 16x the rate of the float32 MFMA) with BOTH operands split x = hi + lo into bf16 planes and three
// passes per product (hi.hi + hi.lo + lo.hi; the dropped lo.lo term is 2^-16 of the product - the accuracy class of the
// bf16x2 GEMMs, where only one operand needs the split).  Per 32-key tile and wave: 24 + 24 MFMAs of ~17 cycles instead of
// 64 + 64 of 32.  K / V tiles are split once, by all 256 threads, while they are staged: K as [key][d] planes (272-byte rows:
// the B fragments of Q.K^T are conflict-free ds_read_b128), V TRANSPOSED as [d][key] planes (80-byte rows) because the B
// operand of P.V needs 8 consecutive KEYS of one head dim per lane - the staging threads of V therefore vary over keys
// within a wave (contiguous 2-byte LDS writes) and pay with 16-byte global reads at a 512-byte stride (L2-resident rows).
// ---------------------------------------------------------------------------------------------------
typedef __bf16 abf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 abf16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void split8(const float (&x)[8], abf16x8_t& hi, abf16x8_t& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const __bf16 h = (__bf16)x[j];
    hi[j] = h;
    lo[j] = (__bf16)(x[j] - (float)h);
  }
}

__global__ __launch_bounds__(256, 2) void attn_prefill_bf16x3_kernel(AttnParams p) {
  constexpr int KT = 32, NB = 2, KROW = 272, VROW = 80, PS = 36;
  __shared__ __attribute__((aligned(16))) char k_hi[KT * KROW];
  __shared__ __attribute__((aligned(16))) char k_lo[KT * KROW];
  __shared__ __attribute__((aligned(16))) char vt_hi[kHeadDim * VROW];
  __shared__ __attribute__((aligned(16))) char vt_lo[kHeadDim * VROW];
  __shared__ __attribute__((aligned(16))) float p_all[4 * 16 * PS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hq = blockIdx.y;
  const int G = p.n_q / p.n_kv, hk = hq / G;
  const int heads = p.n_q + 2 * p.n_kv;
  const int T = p.t, pos0 = p.pos0_dev ? *p.pos0_dev : p.pos0;
  const int qt = gridDim.x - 1 - blockIdx.x;                // heaviest query tiles (most key tiles) first
  const int q0 = qt * 64;
  const int arow = lane & 15, kq = lane >> 4;              // A/B fragment coordinates: row / column, group of 8 K-values
  const int ccol = lane & 15, crow0 = (lane >> 4) * 4;     // C layout
  const float scale2 = 0.08838834764831845f * 1.4426950408889634f;   // d^-1/2 * log2(e): the softmax runs on exp2
  float* p_s = p_all + wave * 16 * PS;

  abf16x8_t q_hi[4], q_lo[4];                                // A fragments of this wave's 16 query rows, 4 K-steps of 32 dims
  {
    int qrow = q0 + wave * 16 + arow;
    if (qrow > T - 1) qrow = T - 1;                         // padded rows compute garbage that is never stored
    const float* qp = p.qkv + ((size_t)qrow * heads + hq) * kHeadDim + kq * 8;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qp + ks * 32), b = *reinterpret_cast<const f32x4*>(qp + ks * 32 + 4);
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      split8(x, q_hi[ks], q_lo[ks]);
    }
  }
  int qpos[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) qpos[r] = pos0 + q0 + wave * 16 + crow0 + r;
  float m_run[4], l_run[4];
  f32x4 o_acc[8];
#pragma unroll
  for (int r = 0; r < 4; ++r) { m_run[r] = -INFINITY; l_run[r] = 0.f; }
#pragma unroll
  for (int db = 0; db < 8; ++db) o_acc[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int last_q = q0 + 63 < T - 1 ? q0 + 63 : T - 1;
  const int kmax = pos0 + last_q;                           // last key any row of this workgroup may see
  const int nkt = kmax / KT + 1;
  const KvLayout kvl{p.table, p.n_kv, p.max_ctx, p.log_block};

  // tile kt+1 is loaded into registers before the MFMAs of tile kt (as in the float32 kernel).
  // K: thread (key = idx >> 5, 4 dims idx & 31): a wave reads two whole key rows.  V: a lane takes the SAME 4 dims of the key
  // pair (2j, 2j+1), j = lane & 15, so that the transposed store is one 4-byte write per dim - the two keys' bf16 values side
  // by side, 16 lanes = 16 consecutive dwords (the first version wrote 2 bytes per lane: 35 % of all LDS cycles were conflicts).
  f32x4 kreg[4], vreg[4];
  const int vj = lane & 15;
  auto load_tile = [&](int kt) {
    const size_t toff = kv_tile_off(kvl, hk, kt * KT);      // first row of the tile (one block-table lookup when paged)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256;
      const int kkey = idx >> 5, kc4 = idx & 31;
      const int kr = kt * KT + kkey <= kmax ? kkey : kmax - kt * KT;    // clamped row inside the tile; masked by key index below
      kreg[i] = *reinterpret_cast<const f32x4*>(p.kc + toff + (size_t)kr * kHeadDim + kc4 * 4);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int vc4 = (tid >> 4) + 16 * i;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int vkey = 2 * vj + h;
        const int vr = kt * KT + vkey <= kmax ? vkey : kmax - kt * KT;
        vreg[2 * i + h] = *reinterpret_cast<const f32x4*>(p.vc + toff + (size_t)vr * kHeadDim + vc4 * 4);
      }
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256;
      const int kkey = idx >> 5, kc4 = idx & 31;
      const float kx[4] = {kreg[i].x, kreg[i].y, kreg[i].z, kreg[i].w};
      abf16x4_t kh, kl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const __bf16 h = (__bf16)kx[e];
        kh[e] = h;
        kl[e] = (__bf16)(kx[e] - (float)h);
      }
      *reinterpret_cast<abf16x4_t*>(k_hi + kkey * KROW + kc4 * 8) = kh;
      *reinterpret_cast<abf16x4_t*>(k_lo + kkey * KROW + kc4 * 8) = kl;
    }
    typedef __bf16 abf16x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int vc4 = (tid >> 4) + 16 * i;
      const float v0[4] = {vreg[2 * i].x, vreg[2 * i].y, vreg[2 * i].z, vreg[2 * i].w};
      const float v1[4] = {vreg[2 * i + 1].x, vreg[2 * i + 1].y, vreg[2 * i + 1].z, vreg[2 * i + 1].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        abf16x2_t h, l;
        h[0] = (__bf16)v0[e]; h[1] = (__bf16)v1[e];
        l[0] = (__bf16)(v0[e] - (float)h[0]); l[1] = (__bf16)(v1[e] - (float)h[1]);
        *reinterpret_cast<abf16x2_t*>(vt_hi + (vc4 * 4 + e) * VROW + vj * 4) = h;
        *reinterpret_cast<abf16x2_t*>(vt_lo + (vc4 * 4 + e) * VROW + vj * 4) = l;
      }
    }
  };
  const int NS = p.n_splits, split = blockIdx.z;
  if (split < nkt) load_tile(split);
  for (int kt = split; kt < nkt; kt += NS) {
    const int k0 = kt * KT;
    __syncthreads();                                        // the previous tile has been consumed by every wave
    store_tile();
    __syncthreads();
    if (kt + NS < nkt) load_tile(kt + NS);
    // the workgroup walks the keys its LAST query row sees; a wave whose 16 rows all lie before this tile has nothing to add
    // (every score masked): wave-uniform skip, the barriers above keep the cadence
    if (k0 > pos0 + q0 + wave * 16 + 15) continue;

    f32x4 s_acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) s_acc[nb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int off = (nb * 16 + arow) * KROW + ks * 64 + kq * 16;
        const abf16x8_t bh = *reinterpret_cast<const abf16x8_t*>(k_hi + off);
        const abf16x8_t bl = *reinterpret_cast<const abf16x8_t*>(k_lo + off);
        s_acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q_lo[ks], bh, s_acc[nb], 0, 0, 0);
        s_acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q_hi[ks], bl, s_acc[nb], 0, 0, 0);
        s_acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q_hi[ks], bh, s_acc[nb], 0, 0, 0);
      }
    }
    // online softmax in the log2 domain: identical to attn_prefill_mfma_kernel (C layout: column = key, 4 rows per lane)
    float mx[4], ps[4], alpha[4], m_ref[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mx[r] = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        float sc = s_acc[nb][r] * scale2;
        if (k0 + nb * 16 + ccol > qpos[r]) sc = -INFINITY;  // causal mask
        s_acc[nb][r] = sc;
        mx[r] = fmaxf(mx[r], sc);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], lane_xor1(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], lane_xor2(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], row_ror4(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], row_ror8(mx[r]));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float m_new = fmaxf(m_run[r], mx[r]);
      m_ref[r] = m_new == -INFINITY ? 0.f : m_new;           // a key split may start on a tile this row cannot see at all
      alpha[r] = __builtin_amdgcn_exp2f(m_run[r] - m_ref[r]);
      m_run[r] = m_new;
      ps[r] = 0.f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float e = __builtin_amdgcn_exp2f(s_acc[nb][r] - m_ref[r]);
        s_acc[nb][r] = e;
        ps[r] += e;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += lane_xor1(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += lane_xor2(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += row_ror4(ps[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[r] += row_ror8(ps[r]);
    // no running maximum of this wave's rows moved (every alpha == 1.0f exactly): the 32 rescaling multiplies would change nothing
    const bool moved = __builtin_amdgcn_ballot_w64(alpha[0] != 1.f || alpha[1] != 1.f || alpha[2] != 1.f || alpha[3] != 1.f) != 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      l_run[r] = l_run[r] * alpha[r] + ps[r];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) p_s[(crow0 + r) * PS + nb * 16 + ccol] = s_acc[nb][r];
    }
    if (moved) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int db = 0; db < 8; ++db) o_acc[db][r] *= alpha[r];
      }
    }
    __builtin_amdgcn_wave_barrier();                        // P is wave private: LDS ops of one wave stay in order
    // P as the A operand of P.V: query row arow, keys kq*8 .. kq*8+7 (two conflict-free ds_read_b128 of the [16][36] tile)
    abf16x8_t p_hi, p_lo;
    {
      const f32x4 a = *reinterpret_cast<const f32x4*>(p_s + arow * PS + kq * 8), b = *reinterpret_cast<const f32x4*>(p_s + arow * PS + kq * 8 + 4);
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      split8(x, p_hi, p_lo);
    }
#pragma unroll
    for (int db = 0; db < 8; ++db) {                        // head dims db*16 .. db*16+15: B fragment = 8 keys of dim db*16 + arow
      const int off = (db * 16 + arow) * VROW + kq * 16;
      const abf16x8_t vh = *reinterpret_cast<const abf16x8_t*>(vt_hi + off);
      const abf16x8_t vl = *reinterpret_cast<const abf16x8_t*>(vt_lo + off);
      o_acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_lo, vh, o_acc[db], 0, 0, 0);
      o_acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_hi, vl, o_acc[db], 0, 0, 0);
      o_acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_hi, vh, o_acc[db], 0, 0, 0);
    }
  }
  // C layout of the output: lane holds head dims db*16 + ccol (db = 0..7) of query rows crow0 + r
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int qrow = q0 + wave * 16 + crow0 + r;
    if (qrow >= T) continue;
    if (NS > 1) {                                           // partial (unnormalised) result of this key split
      const size_t pi = ((size_t)qrow * p.n_q + hq) * NS + split;
#pragma unroll
      for (int db = 0; db < 8; ++db) p.part_o[pi * kHeadDim + db * 16 + ccol] = o_acc[db][r];
      if (ccol == 0) { p.part_ml[pi * 2] = m_run[r] * 0.6931471805599453f; p.part_ml[pi * 2 + 1] = l_run[r]; }   // m back to nats
    } else {
      const float inv = 1.0f / l_run[r];
      const size_t oi = ((size_t)qrow * p.n_q + hq) * kHeadDim;
#pragma unroll
      for (int db = 0; db < 8; ++db) {
#pragma clang fp contract(off)   // lo = split of the ROUNDED product, as chatts_split_bf16x2 of the float32 output would give
        const float v = o_acc[db][r] * inv;
        if (p.out_hi) {
          const __bf16 h = (__bf16)v;
          const size_t at = plane_at(qrow, hq * kHeadDim + db * 16 + ccol, p.n_q * kHeadDim, p.out_tiled);
          p.out_hi[at] = __builtin_bit_cast(uint16_t, h);
          p.out_lo[at] = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)h));
        } else {
          p.out[oi + db * 16 + ccol] = v;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// prefill with K / V planes: the flash loop on TRANSPOSED tiles.  kv_planes_kernel splits the sequence's K / V rows into bf16 hi / lo
// planes ONCE per layer and chunk (attn_prefill_bf16x3_kernel does it once per (query tile, query head): 65 times per tile at T = 798);
// attn_prefill_planes_kernel then computes S^T = K.Q^T and O^T = V^T.P^T, which puts "query = lane & 15" on every operand:
//   * S^T in the C layout gives a lane 8 keys of ONE query: the row maximum is an in-lane maximum + two lane exchanges (xor 16, 32)
//     instead of 4 rows x 4 DPP steps, the row sum stays a per-lane partial until the very end, one alpha per lane;
//   * those 8 probabilities ARE the B fragment of V^T.P^T - P never goes through LDS.  The MFMA's K index is a free choice as long as
//     A and B agree: slot 8 g + j of lane group g means key 4 g + j (j < 4) or 16 + 4 g + (j - 4), and kv_planes_kernel writes the
//     V^T rows in that slot order, so the A fragment is still one 16-byte LDS read;
//   * O^T in the C layout gives a lane 4 consecutive head dims of its query: alpha applies as is, the output is 16-byte stores.
// Same three-pass bf16 split products as the kernel above; the sums run in another order, so
// the two agree to rounding (tests: both against the float64 reference).  Needs the host to know pos0 (plane count) and a free
// workspace; otherwise the kernel above runs.
// Plane layout, per (kv head, 32-key tile) 32 KB: K_hi [32 keys][128], K_lo, V^T_hi [128 dims][32 slots], V^T_lo, every row's 16-byte chunks where LDS wants them (chunk c of key k at
// c ^ (k & 15), chunk c of dim d at c ^ ((d >> 2) & 2)), so that a tile goes to LDS as it lies, by DMA; rows past the last key repeat it (finite values behind the causal mask).
// ---------------------------------------------------------------------------------------------------
// Bound by the round trip to the cache for a few hundred keys, by bytes for thousands.  A thread writes whole chunks and the lanes of a wave write next to each other; 8 bytes of V^T every
// 64 took 5.1 / 8 / 18 us for 223 / 806 / 2048 keys of 8 heads, this 3.7 / 5.8 / 16.6 (with 16-byte loads of V the same).
// one chunk of a tile's planes: 8 dims of a key; 8 slots of a head dim - slot 8 g + j of chunk g is key 4 g + j or (from j = 4 on) 12 + 4 g + j
__device__ __forceinline__ int v_slot_key(int g, int j) { return 4 * g + j + (j < 4 ? 0 : 12); }
__device__ __forceinline__ void store_k_chunk(char* dst, int key, int chunk, const float (&x)[8]) {
  abf16x8_t h, l;
  split8(x, h, l);
  char* to = dst + key * 256 + ((chunk ^ (key & 15)) << 4);
  *reinterpret_cast<abf16x8_t*>(to) = h;
  *reinterpret_cast<abf16x8_t*>(to + 8192) = l;
}
__device__ __forceinline__ void store_v_chunk(char* dst, int d, int g, const float (&x)[8]) {
  abf16x8_t h, l;
  split8(x, h, l);
  char* to = dst + 16384 + d * 64 + ((g ^ ((d >> 2) & 2)) << 4);
  *reinterpret_cast<abf16x8_t*>(to) = h;
  *reinterpret_cast<abf16x8_t*>(to + 8192) = l;
}
// a tile's planes from key4(key, d): K at dims d .. d + 3, and value(key, d): V.  Thread = (key, chunk) and (head dim, chunk), two of each
template <typename K4, typename V1>
__device__ __forceinline__ void store_kv_planes(char* dst, int tid, K4 key4, V1 value) {
  f32x4 kv[2][2];
  float vv[2][8];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) kv[i][h] = key4((tid >> 4) + i * 16, (tid & 15) * 8 + h * 4);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) vv[i][j] = value(v_slot_key(tid & 3, j), (tid >> 2) + i * 64);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float x[8] = {kv[i][0].x, kv[i][0].y, kv[i][0].z, kv[i][0].w, kv[i][1].x, kv[i][1].y, kv[i][1].z, kv[i][1].w};
    store_k_chunk(dst, (tid >> 4) + i * 16, tid & 15, x);
    store_v_chunk(dst, (tid >> 2) + i * 64, tid & 3, vv[i]);
  }
}

__global__ __launch_bounds__(256) void kv_planes_kernel(AttnParams p, int n_keys, uint16_t* planes) {
  constexpr int KT = 32;
  const int tid = threadIdx.x, kt = blockIdx.x, hk = blockIdx.y;
  const KvLayout kvl{p.table, p.n_kv, p.max_ctx, p.log_block};
  const size_t toff = kv_tile_off(kvl, hk, kt * KT);
  char* dst = reinterpret_cast<char*>(planes) + ((size_t)hk * gridDim.x + kt) * (8 * KT * kHeadDim);
  const int last = n_keys - 1 - kt * KT;                    // last valid row inside this tile (>= 0)
  store_kv_planes(dst, tid, [&](int key, int d) { return *reinterpret_cast<const f32x4*>(p.kc + toff + (size_t)(key <= last ? key : last) * kHeadDim + d); },
                  [&](int key, int d) { return p.vc[toff + (size_t)(key <= last ? key : last) * kHeadDim + d]; });
}

// The same from qkv rows that no launch has rotated yet: the chunk's K and V rows go through rope_kv_kernel's work (a wave a row, the same bits) into the cache and, from LDS, into the planes;
// rows before the chunk come from the cache.  The queries are left to attn_prefill_planes_kernel.  Where the qkv projection has no split whose epilogue does it, rope_kv_kernel read and wrote all
// heads and kv_planes_kernel read the cache back: 12.6 + 6.3 us for 798 rows of 40 + 16 heads, 28 + 10 for 2048; here 9 and 12, and the attention 1 more for the queries.  Prompts, ms: 14B of 798 rows
// 36.9 / 36.7, of 2300 105.5 / 104.8, 8B of 1000 24.1 / 23.9.
__global__ __launch_bounds__(256) void rope_kv_planes_kernel(const float* __restrict__ qkv, RopeFuse r, int n_keys, uint16_t* __restrict__ planes) {
  constexpr int KT = 32, LD = kHeadDim + 4;
  __shared__ __attribute__((aligned(16))) float k_s[KT * LD];
  __shared__ __attribute__((aligned(16))) float v_s[KT * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kt = blockIdx.x, hk = blockIdx.y;
  const int heads = r.n_q + 2 * r.n_kv, last = n_keys - 1 - kt * KT;
  const size_t toff = kv_tile_off(r.kvl, hk, kt * KT);
  float k[8][2], v[8][2], c[8], s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int key = wave * 8 + i, kr = key <= last ? key : last, pos = kt * KT + kr, tok = pos - r.pos0;      // (rows past the last key repeat it)
    const float* kp = tok >= 0 ? qkv + ((size_t)tok * heads + r.n_q + hk) * kHeadDim : r.kc + toff + (size_t)kr * kHeadDim;
    const float* vp = tok >= 0 ? qkv + ((size_t)tok * heads + r.n_q + r.n_kv + hk) * kHeadDim : r.vc + toff + (size_t)kr * kHeadDim;
#pragma unroll
    for (int h = 0; h < 2; ++h) { k[i][h] = kp[lane + 64 * h]; v[i][h] = vp[lane + 64 * h]; }
    c[i] = r.cos_tab[(size_t)pos * 64 + lane];
    s[i] = r.sin_tab[(size_t)pos * 64 + lane];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int key = wave * 8 + i, kr = key <= last ? key : last;
    if (kt * KT + kr >= r.pos0) {                           // (uniform)
      norm_rope(k[i][0], k[i][1], r.k_norm_w, r.eps, c[i], s[i], lane);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        k[i][h] = kv_round_f(k[i][h], r.kv_round);
        v[i][h] = kv_round_f(v[i][h], r.kv_round);
        if (key <= last) {
          r.kc[toff + (size_t)kr * kHeadDim + lane + 64 * h] = k[i][h];
          r.vc[toff + (size_t)kr * kHeadDim + lane + 64 * h] = v[i][h];
        }
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) { k_s[key * LD + lane + 64 * h] = k[i][h]; v_s[key * LD + lane + 64 * h] = v[i][h]; }
  }
  __syncthreads();
  store_kv_planes(reinterpret_cast<char*>(planes) + ((size_t)hk * gridDim.x + kt) * (8 * KT * kHeadDim), tid, [&](int key, int d) { return *reinterpret_cast<const f32x4*>(k_s + key * LD + d); },
                  [&](int key, int d) { return v_s[key * LD + d]; });
}

// x[i] += the slabs' values at at[i], slab after slab
template <int N>
__device__ __forceinline__ void sum_slabs(const float* __restrict__ slabs, int sk, size_t plane, const size_t (&at)[N], float (&x)[N]) {
  int s = 0;
  for (; s + 4 <= sk; s += 4) {
    float t[4][N];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < N; ++i) t[u][i] = slabs[(s + u) * plane + at[i]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] += t[u][i];
  }
  for (; s < sk; ++s)
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] += slabs[s * plane + at[i]];
}

// ... and as a split's epilogue (splitk_epilogue_rope_kernel's work; the planes lie behind the slabs): four workgroups a tile and kv head, one for each half of K's keys (a rotation takes a whole
// row) and of V's dims (a chunk takes 8 keys), the others a query head a wave.  One workgroup for a whole tile reads up to 400 KB of slabs by itself: 6 us.  Prompts, us, two launches / here: 8B of 223
// rows 8363 / 8235, 14B of 430 19440 / 19330, 8B of 96 6100 / 6060, 14B of 66 the same.
__global__ __launch_bounds__(256) void rope_epilogue_planes_kernel(const float* __restrict__ slabs, int sk, int m, int n, const float* __restrict__ bias, float* __restrict__ c, int ldc, RopeFuse r,
                                                                   int tiles, uint16_t* __restrict__ planes) {
  constexpr int KT = 32, LDK = kHeadDim + 4, LDV = kHeadDim / 2 + 4;
  __shared__ __attribute__((aligned(16))) float rows_s[16 * LDK > KT * LDV ? 16 * LDK : KT * LDV];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), item = (int)blockIdx.x - tiles * r.n_kv * 4;
  const size_t plane = (size_t)m * n;
  if (item >= 0) {
    const int gw = item * 4 + wave;
    if (gw >= m * r.n_q) return;
    const int tok = gw / r.n_q, h = gw - tok * r.n_q;
    float x[2] = {0.f, 0.f};
    const size_t from = (size_t)tok * n + h * kHeadDim + lane, at[2] = {from, from + 64};
    sum_slabs(slabs, sk, plane, at, x);
    if (bias) { x[0] += bias[h * kHeadDim + lane]; x[1] += bias[h * kHeadDim + lane + 64]; }
    rope_kv_head(x[0], x[1], h, r.pos0 + tok, lane, c + (size_t)tok * ldc + h * kHeadDim, r);
    return;
  }
  const int half = blockIdx.x & 1, is_v = (blockIdx.x >> 1) & 1, kt = (int)(blockIdx.x >> 2) % tiles, hk = (int)(blockIdx.x >> 2) / tiles, last = r.pos0 + m - 1 - kt * KT;
  const int col = (r.n_q + hk + (is_v ? r.n_kv : 0)) * kHeadDim;      // the head's columns
  const size_t toff = kv_tile_off(r.kvl, hk, kt * KT);
  char* dst = reinterpret_cast<char*>(planes) + ((size_t)hk * tiles + kt) * (8 * KT * kHeadDim);
  const bool any = kt * KT + (last < KT - 1 ? last : KT - 1) >= r.pos0;      // of the chunk's rows; those before them come from the cache, rows past the last key repeat it
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  size_t at[8];
  if (is_v) {                                               // 8 keys a wave, 64 dims
    const int d = half * 64 + lane;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = wave * 8 + i, kr = key <= last ? key : last, tok = kt * KT + kr - r.pos0;
      at[i] = (size_t)(tok > 0 ? tok : 0) * n + col + d;
    }
    if (any) sum_slabs(slabs, sk, plane, at, x);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = wave * 8 + i, kr = key <= last ? key : last;
      float* row = r.vc + toff + (size_t)kr * kHeadDim + d;
      if (kt * KT + kr >= r.pos0) {                         // (uniform)
        if (bias) x[i] += bias[col + d];
        x[i] = kv_round_f(x[i], r.kv_round);
        if (key <= last) *row = x[i];
      } else {
        x[i] = *row;
      }
      rows_s[key * LDV + lane] = x[i];
    }
    __syncthreads();
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = rows_s[v_slot_key(tid & 3, j) * LDV + (tid >> 2)];
    store_v_chunk(dst, half * 64 + (tid >> 2), tid & 3, o);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {                             // four keys a wave
    const int key = half * 16 + wave * 4 + i, kr = key <= last ? key : last, tok = kt * KT + kr - r.pos0;
    at[2 * i] = (size_t)(tok > 0 ? tok : 0) * n + col + lane;
    at[2 * i + 1] = at[2 * i] + 64;
  }
  if (any) sum_slabs(slabs, sk, plane, at, x);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k16 = wave * 4 + i, key = half * 16 + k16, kr = key <= last ? key : last, pos = kt * KT + kr;
    float a = x[2 * i], b = x[2 * i + 1], *row = r.kc + toff + (size_t)kr * kHeadDim + lane;
    if (pos >= r.pos0) {                                    // (uniform)
      if (bias) { a += bias[col + lane]; b += bias[col + lane + 64]; }
      norm_rope(a, b, r.k_norm_w, r.eps, r.cos_tab[(size_t)pos * 64 + lane], r.sin_tab[(size_t)pos * 64 + lane], lane);
      a = kv_round_f(a, r.kv_round);
      b = kv_round_f(b, r.kv_round);
      if (key <= last) { row[0] = a; row[64] = b; }
    } else {
      a = row[0];
      b = row[64];
    }
    rows_s[k16 * LDK + lane] = a;
    rows_s[k16 * LDK + lane + 64] = b;
  }
  __syncthreads();
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = rows_s[(tid >> 4) * LDK + (tid & 15) * 8 + j];
  store_k_chunk(dst, half * 16 + (tid >> 4), tid & 15, o);
}

typedef __attribute__((address_space(3))) void* lptr_t;

// the maximum over lanes 16 (32) apart
__device__ __forceinline__ float swap_max16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float swap_max32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// QW waves of QB x 16 queries each, KP parts of the keys: wave (part, w) takes tiles part, part + KP, ... for its queries, and the parts' sums meet in LDS at the end.
// What bounds it, by size: for some hundred rows the chain of a wave's tiles, each ~1 us of LDS reads, products and softmax one after the other (parts shorten the chain; fewer queries a
// workgroup spread the work where CUs would be idle); above that LDS: 16 queries read every tile whole, 32 KB of LDS reads for 48 products (QB = 2: for 96); from some thousand rows on the
// matrix pipe at the rate its power allows.  So: all of K's fragments are asked for at once, V's before the softmax, products run in four chains, tiles come by DMA, one ahead (three
// ahead gained nothing), with one barrier a tile.  With tiles through registers, reads four at a time and 16 queries x one part only, us with kv_planes_kernel (before / now),
// 32 heads: 64 rows 10.1 / 8.1, 223 17.6 / 13.2, 512 32.6 / 24.3, 806 49.0 / 34.8, 2048 145.9 / 122, 64 rows behind 700 keys 42 / 25.6; 40 heads: 806 50 / 41, 2048 174.7 / 142.
// LDS rows have no padding, their 16-byte chunks are XOR-swizzled for ds_read_b128's lane groups ({0-3, 12-15, 20-27}, {4-11, 16-19, 28-31}, ...: every group holds each qi once, with
// g = g0 for eight of them and g0 + 1 for the other eight): each group covers all 64 banks exactly once.
template <int QW, int QB, int KP>
__global__ __launch_bounds__(64 * QW * KP, 2) void attn_prefill_planes_kernel(AttnParams p) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int KT = 32, TILE = 8 * KT * kHeadDim, PIECES = TILE / 1024 / QW;
  extern __shared__ __attribute__((aligned(1024))) char tiles_s[];      // [part][2][K_hi, K_lo, V^T_hi, V^T_lo]
  const int lane = threadIdx.x & 63;
  const int part = __builtin_amdgcn_readfirstlane((int)threadIdx.x / (64 * QW)), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64 % QW);
  char* mine = tiles_s + part * (2 * TILE);
  const int G = p.n_q / p.n_kv;
  // XCD-aware order.  Workgroups go to the 8 XCDs round robin by linear index, each XCD has its own 4 MB L2, and every workgroup
  // streams its kv head's planes (0.8 MB at 798 keys; 233 MB of tile reads per launch in total).  With (query tile, query head) as
  // the grid every XCD saw all kv heads - 6.4 MB through a 4 MB L2.  Here workgroup L works for kv head (L % 8) % n_kv: an XCD keeps
  // ONE kv head's planes (8 / n_kv XCDs share a head), and the items of a head - its G query heads x query tiles, heaviest first - are
  // dealt to those XCDs in turn.  (Measured at 798 keys: the locality itself is worth nothing yet - 43.0 against 42.6 us for a plain
  // head-fastest order - what counts is that the heaviest tiles of ALL heads start first: 47.8 us with (query tile, head) as a 2-D grid.)
  int hk, item;
  if (p.xcd_share > 0) {
    const int c = blockIdx.x & 7;
    hk = c % p.n_kv;
    item = (blockIdx.x >> 3) * p.xcd_share + c / p.n_kv;
    if (item >= G * p.units) return;
  } else {
    hk = (blockIdx.x % p.n_q) / G;
    item = (blockIdx.x / p.n_q) * G + (blockIdx.x % p.n_q) % G;
  }
  const int xi = item / G, hq = hk * G + item % G;
  const int heads = p.n_q + 2 * p.n_kv;
  const int T = p.t, pos0 = p.pos0;
  const int qt = p.units - 1 - xi;                          // heaviest query tiles (most key tiles) first, over ALL heads
  const int q0 = qt * (16 * QB * QW), qw = q0 + wave * (16 * QB);      // first query of the workgroup, of this wave
  const int qi = lane & 15, g = lane >> 4;                  // this lane's query (of the wave's 16) and its group of 8 K-values / 4 C rows
  const float scale2 = 0.08838834764831845f * 1.4426950408889634f;   // d^-1/2 * log2(e): the softmax runs on exp2

  const int last_q = q0 + 16 * QB * QW - 1 < T - 1 ? q0 + 16 * QB * QW - 1 : T - 1;
  const int nkt = (pos0 + last_q) / KT + 1;                 // tiles up to the last key any row of this workgroup may see
  f32x4 q_in[QB][8];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    int qrow = qw + b * 16 + qi;
    if (qrow > T - 1) qrow = T - 1;                         // padded rows compute garbage that is never stored
    const float* qp = p.qkv + ((size_t)qrow * heads + hq) * kHeadDim + g * 8;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) q_in[b][ks] = *reinterpret_cast<const f32x4*>(qp + (ks >> 1) * 32 + (ks & 1) * 4);
  }
  f32x4 turn[QB][8], weight[8];                             // cosines and sines, the norm's weights: only for rows that rope_kv_planes_kernel left as they were
  if (p.cos_tab) {
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      int qrow = qw + b * 16 + qi;
      if (qrow > T - 1) qrow = T - 1;
      const size_t at = (size_t)(pos0 + qrow) * 64 + g * 8;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        turn[b][ks] = *reinterpret_cast<const f32x4*>(p.cos_tab + at + (ks >> 1) * 32 + (ks & 1) * 4);
        turn[b][4 + ks] = *reinterpret_cast<const f32x4*>(p.sin_tab + at + (ks >> 1) * 32 + (ks & 1) * 4);
      }
    }
    if (p.q_norm_w)
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) weight[ks] = *reinterpret_cast<const f32x4*>(p.q_norm_w + g * 8 + (ks >> 1) * 32 + (ks & 1) * 4);
  }
  // a tile of this part, on its way to its place in LDS; past the last one a request returns zeros
  const char* src0 = reinterpret_cast<const char*>(p.kv_planes) + (size_t)hk * p.kv_plane_tiles * TILE;
  auto request = [&](int kt, int at) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(src0 + (size_t)kt * TILE), 0, kt < nkt ? TILE : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lptr_t)(mine + at * TILE + (wave * PIECES + i) * 1024), 16, (wave * PIECES + i) * 1024 + lane * 16, 0, 0, 0);
  };
  __builtin_amdgcn_sched_barrier(0);
  request(part, 0);
  __builtin_amdgcn_sched_barrier(0);
  if (p.cos_tab) {                                          // norm and rotation of 128 dims: 32 in each of four lanes, d and d + 64 in one
#pragma clang fp contract(off)
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      if (p.q_norm_w) {
        float ss = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss += q_in[b][ks][e] * q_in[b][ks][e];
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        const float rstd = rsqrtf(ss / (float)kHeadDim + p.eps);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
          for (int e = 0; e < 4; ++e) q_in[b][ks][e] = weight[ks][e] * (q_in[b][ks][e] * rstd);
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = q_in[b][ks][e], y = q_in[b][ks + 4][e], c = turn[b][ks][e], sn = turn[b][4 + ks][e];
          q_in[b][ks][e] = x * c - y * sn;
          q_in[b][ks + 4][e] = y * c + x * sn;
        }
    }
  }
  abf16x8_t q_hi[QB][4], q_lo[QB][4];                        // B fragments of Q^T: query qi, dims ks*32 + g*8 .. +7
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f32x4 v0 = q_in[b][2 * ks], v1 = q_in[b][2 * ks + 1];
      const float x[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
      split8(x, q_hi[b][ks], q_lo[b][ks]);
    }
  const int qpos = pos0 + qw + qi;
  float m_run[QB], l_part[QB];                              // l_part: this lane's 8 slots only; the four groups meet after the loop
  f32x4 o_acc[QB][8];                                       // O^T: head dims db*16 + 4 g + r of query qi
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    m_run[b] = -INFINITY;
    l_part[b] = 0.f;
#pragma unroll
    for (int db = 0; db < 8; ++db) o_acc[b][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }

  auto tile = [&](int kt, int at) __attribute__((always_inline)) {
    const int k0 = kt * KT;
    if (kt >= nkt || k0 > pos0 + qw + 16 * QB - 1) return;      // no tile / every score of this wave masked: wave-uniform skip
    const char* base = mine + at * TILE;
    abf16x8_t fh[8], fl[8];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const char* from = base + (nb * 16 + qi) * 256 + (((ks * 4 + g) ^ qi) << 4);
        fh[ks * 2 + nb] = *reinterpret_cast<const abf16x8_t*>(from);
        fl[ks * 2 + nb] = *reinterpret_cast<const abf16x8_t*>(from + 8192);
      }
    __builtin_amdgcn_sched_barrier(0);
    constexpr int NC = QB > 1 ? 1 : 2;                      // S^T: keys k0 + nb*16 + 4 g + r, query qi; in four chains of products
    f32x4 s_acc[QB][2][NC];
#pragma unroll
    for (int b = 0; b < QB; ++b)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int c = 0; c < NC; ++c) s_acc[b][nb][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) {
            f32x4& to = s_acc[b][nb][t == 1 ? NC - 1 : 0];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t == 2 ? fl[ks * 2 + nb] : fh[ks * 2 + nb], t == 0 ? q_lo[b][ks] : q_hi[b][ks], to, 0, 0, 0);
          }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < 8; ++db) {                        // head dims db*16 .. db*16+15: A fragment = 8 slots of dim db*16 + qi; under way while the softmax runs
      const char* from = base + 16384 + (db * 16 + qi) * 64 + ((g ^ ((qi >> 2) & 2)) << 4);
      fh[db] = *reinterpret_cast<const abf16x8_t*>(from);
      fl[db] = *reinterpret_cast<const abf16x8_t*>(from + 8192);
    }
    __builtin_amdgcn_sched_barrier(0);
    const bool diag = k0 + KT - 1 > pos0 + qw;  // wave-uniform: only such a tile holds keys some query of this wave cannot see
    abf16x8_t p_hi[QB], p_lo[QB];                            // B fragments of P^T: slots 8 g .. 8 g + 7 of query qi
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float e[8];
      float mx = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float sc = s_acc[b][nb][0][r];
          if (NC > 1) sc += s_acc[b][nb][NC - 1][r];
          sc *= scale2;
          if (diag && k0 + nb * 16 + 4 * g + r > qpos + b * 16) sc = -INFINITY;   // causal mask
          e[nb * 4 + r] = sc;
          mx = fmaxf(mx, sc);
        }
      }
      mx = swap_max16(mx);
      mx = swap_max32(mx);
      const float m_new = fmaxf(m_run[b], mx);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run[b] - m_ref);
      m_run[b] = m_new;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[j] = __builtin_amdgcn_exp2f(e[j] - m_ref);
        ps += e[j];
      }
      l_part[b] = l_part[b] * alpha + ps;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {    // some running maximum of this wave moved
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          o_acc[b][db].x *= alpha; o_acc[b][db].y *= alpha; o_acc[b][db].z *= alpha; o_acc[b][db].w *= alpha;
        }
      }
      split8(e, p_hi[b], p_lo[b]);
    }
    constexpr int ND = 4 / QB;                               // (four chains here, too)
#pragma unroll
    for (int d0 = 0; d0 < 8; d0 += ND) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int db = d0; db < d0 + ND; ++db)
#pragma unroll
          for (int b = 0; b < QB; ++b)
            o_acc[b][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t == 1 ? fl[db] : fh[db], t == 0 ? p_lo[b] : p_hi[b], o_acc[b][db], 0, 0, 0);
    }
  };
  for (int k0 = 0, at = 0; k0 < nkt; k0 += KP, at ^= 1) {     // (the same for all parts: they meet at the barriers)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                            // all of this tile has landed, and the tile before it has been consumed by every wave
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    request(k0 + part + KP, at ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    tile(k0 + part, at);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // (no request outlives its LDS)
  if constexpr (KP > 1) {                                    // part 0 has seen key 0: its maximum is that of a score unless there is none
    f32x4* sums = reinterpret_cast<f32x4*>(tiles_s);         // [part - 1][wave][block][o 0 .. 7, (m, l)][lane]
    __syncthreads();
    if (part > 0) {
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        f32x4* to = sums + (((part - 1) * QW + wave) * QB + b) * (9 * 64) + lane;
#pragma unroll
        for (int db = 0; db < 8; ++db) to[db * 64] = o_acc[b][db];
        to[8 * 64] = (f32x4){m_run[b], l_part[b], 0.f, 0.f};
      }
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int j = 0; j < KP - 1; ++j)
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const f32x4* from = sums + ((j * QW + wave) * QB + b) * (9 * 64) + lane;
        const f32x4 ml = from[8 * 64];
        const float m_new = fmaxf(m_run[b], ml.x), m_ref = m_new == -INFINITY ? 0.f : m_new;
        const float wa = __builtin_amdgcn_exp2f(m_run[b] - m_ref), wb = __builtin_amdgcn_exp2f(ml.x - m_ref);
        m_run[b] = m_new;
        l_part[b] = l_part[b] * wa + ml.y * wb;
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          const f32x4 o = from[db * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) o_acc[b][db][e] = o_acc[b][db][e] * wa + o[e] * wb;
        }
      }
  }
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    float l = l_part[b] + __shfl_xor(l_part[b], 16);
    l += __shfl_xor(l, 32);
    const int qrow = qw + b * 16 + qi;
    if (qrow >= T) continue;
    const float inv = 1.0f / l;
    const size_t oi = ((size_t)qrow * p.n_q + hq) * kHeadDim + 4 * g;
#pragma unroll
    for (int db = 0; db < 8; ++db) {
#pragma clang fp contract(off)   // lo = split of the ROUNDED product, as chatts_split_bf16x2 of the float32 output would give
      const float v[4] = {o_acc[b][db].x * inv, o_acc[b][db].y * inv, o_acc[b][db].z * inv, o_acc[b][db].w * inv};
      if (p.out_hi) {
        abf16x4_t h, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const __bf16 hh = (__bf16)v[j];
          h[j] = hh;
          lo[j] = (__bf16)(v[j] - (float)hh);
        }
        const size_t at_o = plane_at(qrow, hq * kHeadDim + 4 * g + db * 16, p.n_q * kHeadDim, p.out_tiled);
        *reinterpret_cast<abf16x4_t*>(p.out_hi + at_o) = h;
        *reinterpret_cast<abf16x4_t*>(p.out_lo + at_o) = lo;
      } else {
        *reinterpret_cast<f32x4*>(p.out + oi + db * 16) = (f32x4){v[0], v[1], v[2], v[3]};
      }
    }
  }
#endif
}

// The form, by how the workgroups fill the CUs.  Two waves of queries, two parts of the keys: while there is a CU for every workgroup.  Four waves and two parts: as long as all tiles
// together would take the CUs no longer than the heaviest workgroup takes by itself (the causal mask leaves the others less).  Then one part, two workgroups a CU, 16 or 32 queries a wave: the smaller
// estimate of the larger of all tiles spread over the CUs, the heaviest workgroup's, and, where there are more workgroups than places, two that follow each other in one place (us a tile: 0.75
// spread, 1.05 alone for 16 queries, 1.3 and 1.9 for 32).  us of the four forms: 223 rows of 32 heads 13.2 / 14.1 / 14.7 / 20.2, 512 25.2 / 24.3 / 27.2 / 37.5, 806 48.7 / 34.8 / 40.4 / 55,
// 1400 110 / 78 / 69 / 94, 4000 - / - / 415 / 383; 40 heads: 650 45 / 33.9 / 34.4 / 45.7, 806 60 / 44.2 / 41.4 / 57, 2048 260 / 166 / 150 / 143, 2048 behind 2048 - / - / 410 / 429,
// 2600 behind 2048 - / - / 576 / 513.
enum { PLANES_2X2, PLANES_4X2, PLANES_4X1, PLANES_4X1_32 };
static int prefill_planes_form(int t, int pos0, int n_q, int cus) {
  // tiles of the workgroups of the i-th heaviest tile of q queries
  auto tiles = [&](int q, int i) { return (pos0 + (i == 0 ? t : ((t + q - 1) / q - i) * q) + 31) / 32; };
  auto all = [&](int q) {
    double sum = 0;
    for (int i = 0; i < (t + q - 1) / q; ++i) sum += tiles(q, i);
    return sum * n_q;
  };
  auto estimate = [&](int q, double spread, double alone) {
    const double a = all(q) / cus * spread, b = tiles(q, 0) * alone;
    const int first = 2 * cus / n_q;
    const double c = (t + q - 1) / q > first ? 2 * tiles(q, first) * 2 * spread : 0;
    return a > b ? (a > c ? a : c) : (b > c ? b : c);
  };
  if (n_q * ((t + 31) / 32) <= cus) return PLANES_2X2;
  if (all(64) <= (double)cus * tiles(64, 0)) return PLANES_4X2;
  return estimate(128, 1.3, 1.9) < estimate(64, 0.75, 1.05) ? PLANES_4X1_32 : PLANES_4X1;
}

template <int QW, int QB, int KP>
static int launch_prefill_planes(AttnParams& p, hipStream_t s) {
  constexpr int lds = KP * 2 * 4 * 32 * kHeadDim * (int)sizeof(uint16_t);
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_planes_kernel<QW, QB, KP>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "attention: cannot reserve %d KB of LDS: %s", lds / 1024, hipGetErrorString(e));
    configured = true;
  }
  const int G = p.n_q / p.n_kv;
  p.units = (p.t + 16 * QB * QW - 1) / (16 * QB * QW);
  const int grid = p.xcd_share ? 8 * ((G * p.units + p.xcd_share - 1) / p.xcd_share) : p.n_q * p.units;
  hipLaunchKernelGGL((attn_prefill_planes_kernel<QW, QB, KP>), dim3(grid), dim3(64 * QW * KP), lds, s, p);
  return CHATTS_OK;
}

// merge the split partials of attn_rows_kernel (splits that saw no tile hold m = -inf, l = 0)
__global__ __launch_bounds__(128) void attn_combine_kernel(AttnParams p) {
  const int hq = blockIdx.x, row = blockIdx.y, d = threadIdx.x;
  const size_t base = ((size_t)row * p.n_q + hq) * p.n_splits;
  float M = -INFINITY;
  for (int s = 0; s < p.n_splits; ++s) M = fmaxf(M, p.part_ml[(base + s) * 2]);
  float num = 0.f, den = 0.f;
  for (int s = 0; s < p.n_splits; ++s) {
    const float m = p.part_ml[(base + s) * 2];
    if (m == -INFINITY) continue;
    const float w = expf(m - M);
    num = fmaf(w, p.part_o[(base + s) * kHeadDim + d], num);
    den = fmaf(w, p.part_ml[(base + s) * 2 + 1], den);
  }
  const size_t oi = ((size_t)row * p.n_q + hq) * kHeadDim + d;
  const float v = num / den;
  if (p.out_hi) {                                 // the o_proj operand format, written where the value is made
    const __bf16 h = (__bf16)v;
    p.out_hi[oi] = __builtin_bit_cast(uint16_t, h);
    p.out_lo[oi] = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)h));
  } else {
    p.out[oi] = v;
  }
}

// Combine of the key-split MFMA prefill path (n_splits <= 4): one workgroup per query row, every thread merges float4s of
// the row's n_q x 128 outputs (the (head, row)-per-workgroup kernel above costs 16 us at T = 798 just in launch count).
__global__ __launch_bounds__(256) void attn_combine_rows_kernel(AttnParams p) {
  const int row = blockIdx.x, NS = p.n_splits;
  const int per_row = p.n_q * (kHeadDim / 4);
  for (int q = threadIdx.x; q < per_row; q += 256) {
    const int hq = q / (kHeadDim / 4), d4 = (q % (kHeadDim / 4)) * 4;
    const size_t base = ((size_t)row * p.n_q + hq) * NS;
    float M = -INFINITY;
    for (int s = 0; s < NS; ++s) M = fmaxf(M, p.part_ml[(base + s) * 2]);
    f32x4 num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
    for (int s = 0; s < NS; ++s) {
      const float m = p.part_ml[(base + s) * 2];
      if (m == -INFINITY) continue;
      const float w = expf(m - M);
      const f32x4 o = *reinterpret_cast<const f32x4*>(p.part_o + (base + s) * kHeadDim + d4);
      num.x = fmaf(w, o.x, num.x); num.y = fmaf(w, o.y, num.y); num.z = fmaf(w, o.z, num.z); num.w = fmaf(w, o.w, num.w);
      den = fmaf(w, p.part_ml[(base + s) * 2 + 1], den);
    }
    const size_t oi = ((size_t)row * p.n_q + hq) * kHeadDim + d4;
    const float v[4] = {num.x / den, num.y / den, num.z / den, num.w / den};
    if (p.out_hi) {
      typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));
      bf16x4v hv, lv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const __bf16 h = (__bf16)v[j];
        hv[j] = h;
        lv[j] = (__bf16)(v[j] - (float)h);
      }
      const size_t at = plane_at(row, hq * kHeadDim + d4, p.n_q * kHeadDim, p.out_tiled);
      *reinterpret_cast<bf16x4v*>(p.out_hi + at) = hv;
      *reinterpret_cast<bf16x4v*>(p.out_lo + at) = lv;
    } else {
      *reinterpret_cast<f32x4*>(p.out + oi) = (f32x4){v[0], v[1], v[2], v[3]};
    }
  }
}

}  // namespace chatts

using namespace chatts;

extern "C" size_t chatts_attn_workspace(int t, int n_q, int n_splits) {
  if (n_splits < 1) n_splits = 1;      // the decode kernel always emits partials, even with one slot
  return (size_t)t * n_q * n_splits * (kHeadDim + 2) * sizeof(float);
}

static int bind_workspace(AttnParams& p, void* workspace, size_t workspace_bytes) {
  const size_t need = chatts_attn_workspace(p.t, p.n_q, p.n_splits);
  CHATTS_REQUIRE(workspace && workspace_bytes >= need, CHATTS_E_WORKSPACE,
                 "attention: needs %zu workspace bytes, got %zu", need, workspace_bytes);
  p.part_o = reinterpret_cast<float*>(workspace);
  p.part_ml = p.part_o + (size_t)p.t * p.n_q * p.n_splits * kHeadDim;
  return CHATTS_OK;
}

// cache -> kernel parameters; the block-paged form is validated here (every entry point goes through this)
static int bind_cache(AttnParams& p, const ChattsKvCache* cache) {
  p.kc = cache->k; p.vc = cache->v; p.max_ctx = cache->max_ctx;
  p.table = cache->block_table; p.log_block = 0; p.table_stride = cache->table_stride;
  if (cache->block_table) {
    p.log_block = kv_log_block(cache->block_size);
    CHATTS_REQUIRE(p.log_block > 0, CHATTS_E_BADARG, "attention: block_size %d is not a power of two in 64..32768", cache->block_size);
    CHATTS_REQUIRE(cache->max_ctx % cache->block_size == 0, CHATTS_E_BADARG,
                   "attention: a paged cache of %d positions needs whole blocks of %d", cache->max_ctx, cache->block_size);
  }
  return CHATTS_OK;
}

namespace chatts {
int attention_impl(const float* qkv, int t, int n_q, int n_kv, int pos0, const int32_t* pos0_dev, const ChattsKvCache* cache, float* out,
                   uint16_t* out_hi, uint16_t* out_lo, int n_splits, void* workspace, size_t workspace_bytes, chatts_stream_t stream, int out_tiled = 0, const RopeFuse* rope = nullptr,
                   const uint16_t* planes = nullptr);

// The attention on K / V planes: the positions known here, keys in one split, the caller's workspace free and large enough for the planes
bool prefill_on_planes(int t, int n_kv, int pos0, const int32_t* pos0_dev, bool out_planes, int n_splits, const void* workspace, size_t workspace_bytes) {
  return opt_get(OPT_ATTN_BF16X3, 1) != 0 && opt_get(OPT_ATTN_PLANES, 1) != 0 && (opt_get(OPT_ATTN_ROWS, 0) == 0 || out_planes) && !pos0_dev && n_splits == 1 && t >= 64 && workspace &&
         workspace_bytes >= prefill_plane_bytes(pos0 + t, n_kv) && ((uintptr_t)workspace % 16) == 0;
}
int launch_rope_epilogue_planes(const float* slabs, int sk, int m, int n, const float* bias, float* c, int ldc, const RopeFuse& r, uint16_t* planes, hipStream_t s) {
  const int tiles = (r.pos0 + m + 31) / 32;
  hipLaunchKernelGGL(rope_epilogue_planes_kernel, dim3(tiles * r.n_kv * 4 + (m * r.n_q + 3) / 4), dim3(256), 0, s, slabs, sk, m, n, bias, c, ldc, r, tiles, planes);
  CHATTS_CHECK_LAUNCH("rope_epilogue_planes");
  return CHATTS_OK;
}
// chatts_rope_kv_write and chatts_attention, in one launch fewer and without the queries' way through memory where the planes' writer can do the keys' and values' part
int rope_attention_impl(float* qkv, int t, int n_q, int n_kv, const float* q_norm_w, const float* k_norm_w, float norm_eps, const float* cos_tab, const float* sin_tab, int pos0,
                        const int32_t* pos0_dev, const ChattsKvCache* cache, float* out, uint16_t* out_hi, uint16_t* out_lo, int n_splits, void* workspace, size_t workspace_bytes,
                        chatts_stream_t stream, int out_tiled) {
  if (t > 0 && opt_get(OPT_ROPE_FUSE, 1) != 0 && prefill_on_planes(t, n_kv, pos0, pos0_dev, out_hi != nullptr, n_splits, workspace, workspace_bytes) &&
      (((uintptr_t)cos_tab | (uintptr_t)sin_tab | (uintptr_t)q_norm_w) % 16) == 0) {
    RopeFuse r;
    if (const int rc = rope_fuse_prepare(t, n_q, n_kv, q_norm_w, k_norm_w, norm_eps, cos_tab, sin_tab, pos0, nullptr, cache, &r)) return rc;
    return attention_impl(qkv, t, n_q, n_kv, pos0, nullptr, cache, out, out_hi, out_lo, n_splits, workspace, workspace_bytes, stream, out_tiled, &r);
  }
  if (const int rc = chatts_rope_kv_write(qkv, t, n_q, n_kv, q_norm_w, k_norm_w, norm_eps, cos_tab, sin_tab, pos0, pos0_dev, cache, stream)) return rc;
  return attention_impl(qkv, t, n_q, n_kv, pos0, pos0_dev, cache, out, out_hi, out_lo, n_splits, workspace, workspace_bytes, stream, out_tiled);
}
}  // namespace chatts

extern "C" int chatts_attention(const float* qkv, int t, int n_q, int n_kv, int pos0, const int32_t* pos0_dev,
                                const ChattsKvCache* cache, float* out, int n_splits, void* workspace,
                                size_t workspace_bytes, chatts_stream_t stream) {
  return chatts::attention_impl(qkv, t, n_q, n_kv, pos0, pos0_dev, cache, out, nullptr, nullptr, n_splits, workspace,
                                workspace_bytes, stream);
}

// chatts_attention with an optional plane output (internal: the decoder's prefill feeds o_proj's LDS-DMA GEMM directly).
// Planes are written by the MFMA kernel / its combine only (t >= 16, n_splits <= 4): the caller checks that.
int chatts::attention_impl(const float* qkv, int t, int n_q, int n_kv, int pos0, const int32_t* pos0_dev,
                           const ChattsKvCache* cache, float* out, uint16_t* out_hi, uint16_t* out_lo, int n_splits,
                           void* workspace, size_t workspace_bytes, chatts_stream_t stream, int out_tiled, const RopeFuse* rope, const uint16_t* planes) {
  CHATTS_REQUIRE(t >= 0 && n_q > 0 && n_kv > 0 && n_splits >= 1 && n_splits <= kMaxSlots, CHATTS_E_BADARG,
                 "attention: bad sizes");
  if (t == 0) return CHATTS_OK;
  CHATTS_REQUIRE(qkv && (out || (out_hi && out_lo)) && cache && cache->k && cache->v, CHATTS_E_BADARG, "attention: null pointer");
  CHATTS_REQUIRE(!out_hi || (t >= 16 && n_splits <= 4), CHATTS_E_BADARG, "attention: plane output needs the MFMA path");
  CHATTS_REQUIRE(n_q % n_kv == 0 && n_q / n_kv <= kMaxGroup, CHATTS_E_SHAPE,
                 "attention: GQA group %d/%d unsupported (max %d)", n_q, n_kv, kMaxGroup);
  if (!pos0_dev)
    CHATTS_REQUIRE(pos0 >= 0 && pos0 + t <= cache->max_ctx, CHATTS_E_SHAPE, "attention: positions exceed the cache");
  AttnParams p{};
  p.qkv = qkv; p.out = out; p.pos0_dev = pos0_dev; p.pos0 = pos0;
  p.t = t; p.n_q = n_q; p.n_kv = n_kv; p.n_splits = n_splits;
  if (const int rc = bind_cache(p, cache)) return rc;
  p.out_hi = out_hi; p.out_lo = out_lo; p.out_tiled = out_tiled;
  if (n_splits > 1) {
    const int rc = bind_workspace(p, workspace, workspace_bytes);
    if (rc) return rc;
  }
  const bool force_rows = opt_get(OPT_ATTN_ROWS, 0) != 0;   // debugging aid: VALU kernel for every T
  // rope / planes: prefill_on_planes has been asked, and nothing else can take these rows (not again: options may change beside a running call)
  const bool on_planes = rope || planes;
  if (t >= 16 && n_splits <= 4 && (!force_rows || out_hi || on_planes)) {
    // (64-key tiles were measured too: 155 us vs 148 us at T = 798 - the per-tile work is not what is slow)
    const int bf16x3 = opt_get(OPT_ATTN_BF16X3, 1);      // 0: the float32-MFMA kernel
    // K / V split into bf16 planes once (kv_planes_kernel) when the caller's workspace is free (one key split) and holds them
    const int n_keys = pos0 + t, tiles = (n_keys + 31) / 32;
    if (on_planes || prefill_on_planes(t, n_kv, pos0, pos0_dev, out_hi != nullptr, n_splits, workspace, workspace_bytes)) {
      uint16_t* pl = static_cast<uint16_t*>(workspace);
      if (planes) {      // (launch_rope_epilogue_planes has written them)
        pl = const_cast<uint16_t*>(planes);
      } else if (rope) {      // (rope_attention_impl: rows of qkv as the projection left them)
        p.q_norm_w = rope->q_norm_w; p.cos_tab = rope->cos_tab; p.sin_tab = rope->sin_tab; p.eps = rope->eps;
        hipLaunchKernelGGL(rope_kv_planes_kernel, dim3(tiles, n_kv), dim3(256), 0, as_stream(stream), qkv, *rope, n_keys, pl);
      } else {
        hipLaunchKernelGGL(kv_planes_kernel, dim3(tiles, n_kv), dim3(256), 0, as_stream(stream), p, n_keys, pl);
      }
      CHATTS_CHECK_LAUNCH("kv_planes");
      p.kv_planes = pl; p.kv_plane_tiles = tiles;
      const bool xcd_on = opt_get(OPT_ATTN_XCD, 1) != 0;
      p.xcd_share = xcd_on && n_kv <= 8 && 8 % n_kv == 0 ? 8 / n_kv : 0;
      int rc;
      switch (prefill_planes_form(t, pos0, n_q, device_cus())) {
        case PLANES_2X2: rc = launch_prefill_planes<2, 1, 2>(p, as_stream(stream)); break;
        case PLANES_4X2: rc = launch_prefill_planes<4, 1, 2>(p, as_stream(stream)); break;
        case PLANES_4X1: rc = launch_prefill_planes<4, 1, 1>(p, as_stream(stream)); break;
        default: rc = launch_prefill_planes<4, 2, 1>(p, as_stream(stream));
      }
      if (rc) return rc;
    } else if (bf16x3) hipLaunchKernelGGL(attn_prefill_bf16x3_kernel, dim3((t + 63) / 64, n_q, n_splits), dim3(256), 0, as_stream(stream), p);
    else hipLaunchKernelGGL(attn_prefill_mfma_kernel<32>, dim3((t + 63) / 64, n_q, n_splits), dim3(256), 0, as_stream(stream), p);
    CHATTS_CHECK_LAUNCH("attn_prefill_mfma");
    if (n_splits > 1) {
      hipLaunchKernelGGL(attn_combine_rows_kernel, dim3(t), dim3(256), 0, as_stream(stream), p);
      CHATTS_CHECK_LAUNCH("attn_combine_rows");
    }
    return CHATTS_OK;
  }
  hipLaunchKernelGGL(attn_rows_kernel, dim3(n_kv, t, n_splits), dim3(256), 0, as_stream(stream), p);
  CHATTS_CHECK_LAUNCH("attn_rows");
  if (n_splits > 1) {
    hipLaunchKernelGGL(attn_combine_kernel, dim3(n_q, t), dim3(128), 0, as_stream(stream), p);
    CHATTS_CHECK_LAUNCH("attn_combine");
  }
  return CHATTS_OK;
}

namespace chatts {
// Which qkv projections of 2 .. 16 rows leave their splits to the attention: those of two to eight, for groups of four and five heads.  Every wave of every slot reads them, and still no
// measured cell lost: us a layer that the launch of their own cost more, contexts 100 / 400 / 1200 / 2000 / 4000, 16 rows, all slots taken:
//   the projection's own number of splits: ChatTS-14B bf16 2.2 / 1.9 / 1.2 / 1.5 / 1.4, fp8 2.5 / 2.5 / 2.0 / 2.5 / 2.6;   ChatTS-8B bf16 2.4 / 1.9 / 1.4 / 1.6 / 1.7, int8 2.1 / 1.8 / 1.3 / 1.7 / 1.5
//   ChatTS-14B bf16, two 2.2 / 1.8 / 2.0 / 2.3 / 2.5, five 2.2 / 1.7 / 1.2 / 1.5 / 1.2, eight 2.1 / 1.2 / 0.8 / 1.0 / 1.0;   ChatTS-8B int8, six 2.1 / 1.0 / 0.6 / 0.8 / 0.9, eight 2.6 / 1.2 / 0.7 / 0.9 / 0.9
// 5 and 8 (8-bit weights), 9 and 12 rows 0.8 to 2.4; half of ChatTS-14B's heads in fp8, 9 and 16 rows 1.1 to 1.5 (the other shards of two, four and eight ranks leave none).
// Other groups keep it, too: the forms whose heads are counted at run time read a head behind a branch, so a head's splits would be a round trip each.  Instances for them are not measured.
bool attn_takes_splits(int n_q, int n_kv) { return n_kv > 0 && (n_q == 4 * n_kv || n_q == 5 * n_kv) && opt_get(OPT_ATTN_EXACT, 1) != 0; }
// chatts_attention_decode_batched with an optional plane output (internal: the decoder's batched step feeds o_proj's
// weight-streaming kernel directly from the combine)
int attention_decode_batched_impl(const float* qkv_raw, int batch, int n_q, int n_kv, const float* q_norm_w,
                                  const float* k_norm_w, float norm_eps, const float* cos_tab, const float* sin_tab, int pos,
                                  const int32_t* pos_dev, const ChattsKvCache* cache, size_t seq_stride, float* out,
                                  uint16_t* out_hi, uint16_t* out_lo, int n_splits, void* workspace, size_t workspace_bytes,
                                  chatts_stream_t stream, const SplitSums* in) {
  CHATTS_REQUIRE(batch >= 1 && n_q > 0 && n_kv > 0 && n_splits >= 1 && n_splits <= kMaxSlots, CHATTS_E_BADARG,
                 "attention_decode: bad sizes (batch >= 1, 1 <= n_splits <= %d)", kMaxSlots);
  CHATTS_REQUIRE(qkv_raw && (out || (out_hi && out_lo)) && cos_tab && sin_tab && cache && cache->k && cache->v, CHATTS_E_BADARG,
                 "attention_decode: null pointer");
  CHATTS_REQUIRE((q_norm_w == nullptr) == (k_norm_w == nullptr), CHATTS_E_BADARG,
                 "attention_decode: q_norm and k_norm must both be set or both be null");
  CHATTS_REQUIRE(n_q % n_kv == 0 && n_q / n_kv <= kMaxGroup, CHATTS_E_SHAPE,
                 "attention: GQA group %d/%d unsupported (max %d)", n_q, n_kv, kMaxGroup);
  CHATTS_REQUIRE(batch == 1 || pos_dev, CHATTS_E_BADARG, "attention_decode: batch > 1 needs per-sequence positions on the device");
  if (!pos_dev)
    CHATTS_REQUIRE(pos >= 0 && pos < cache->max_ctx, CHATTS_E_SHAPE, "attention_decode: position exceeds the cache");
  AttnParams p{};
  p.qkv = qkv_raw; p.out = out; p.pos0_dev = pos_dev; p.pos0 = pos;
  p.t = batch; p.n_q = n_q; p.n_kv = n_kv; p.n_splits = n_splits;
  if (const int rc = bind_cache(p, cache)) return rc;
  p.q_norm_w = q_norm_w; p.k_norm_w = k_norm_w; p.cos_tab = cos_tab; p.sin_tab = sin_tab; p.eps = norm_eps;
  p.seq_stride = seq_stride; p.out_hi = out_hi; p.out_lo = out_lo; p.kv_round = kv_round_mode();
  const int rc = bind_workspace(p, workspace, workspace_bytes);
  if (rc) return rc;
  const dim3 grid(n_kv, n_splits, batch);
  const dim3 wave(64);
  if (in) {
    CHATTS_REQUIRE(attn_takes_splits(n_q, n_kv) && in->sk >= 1 && in->sk <= kMostSplitSums && in->n == (n_q + 2 * n_kv) * kHeadDim, CHATTS_E_SHAPE, "attention_decode: %d splits of %d columns", in->sk, in->n);
    p.qkv = in->slabs; p.qkv_plane = in->plane; p.qkv_splits = in->sk; p.qkv_scale = in->scale; p.qkv_bias = in->bias;
#define CHATTS_ATTN_IN(G, S) hipLaunchKernelGGL((attn_decode_kernel<G, true, false, S>), grid, wave, 0, as_stream(stream), p)
    switch ((n_q / n_kv == 5 ? 8 : 0) + (in->sk <= 4 ? 0 : in->sk - 4 < 2 ? 1 : 2)) {
      case 0: CHATTS_ATTN_IN(4, 4); break;
      case 1: CHATTS_ATTN_IN(4, 5); break;
      case 2: CHATTS_ATTN_IN(4, kMostSplitSums); break;
      case 8: CHATTS_ATTN_IN(5, 4); break;
      case 9: CHATTS_ATTN_IN(5, 5); break;
      default: CHATTS_ATTN_IN(5, kMostSplitSums); break;
    }
#undef CHATTS_ATTN_IN
  }
  // registers sized for the group (every head's arithmetic is the same in all instantiations); the groups of the shipped models
  // (Qwen2.5-14B: 5, Qwen3-8B: 4) get the form with the head count known to the compiler; option ATTN_EXACT=0: the run-time form
  const bool exact = opt_get(OPT_ATTN_EXACT, 1) != 0;
  if (!in) switch (n_q / n_kv) {
    case 4: if (exact) { hipLaunchKernelGGL((attn_decode_kernel<4, true>), grid, wave, 0, as_stream(stream), p); break; }
    case 1: case 2: case 3: hipLaunchKernelGGL((attn_decode_kernel<4, false>), grid, wave, 0, as_stream(stream), p); break;
    case 5: if (exact) hipLaunchKernelGGL((attn_decode_kernel<5, true>), grid, wave, 0, as_stream(stream), p);
            else hipLaunchKernelGGL((attn_decode_kernel<5, false>), grid, wave, 0, as_stream(stream), p);
            break;
    case 6: hipLaunchKernelGGL((attn_decode_kernel<6, false>), grid, wave, 0, as_stream(stream), p); break;
    default: hipLaunchKernelGGL((attn_decode_kernel<4, false, true>), dim3(n_kv, 2 * n_splits, batch), wave, 0, as_stream(stream), p); break;
  }
  CHATTS_CHECK_LAUNCH("attn_decode");
  const dim3 heads(n_q, batch), two(128);
  if (n_splits <= 16) hipLaunchKernelGGL(attn_decode_combine_kernel<16>, heads, two, 0, as_stream(stream), p);
  else if (n_splits <= 32) hipLaunchKernelGGL(attn_decode_combine_kernel<32>, heads, two, 0, as_stream(stream), p);
  else hipLaunchKernelGGL(attn_decode_combine_kernel<64>, heads, two, 0, as_stream(stream), p);
  CHATTS_CHECK_LAUNCH("attn_decode_combine");
  return CHATTS_OK;
}
}  // namespace chatts

extern "C" int chatts_attention_decode_batched(const float* qkv_raw, int batch, int n_q, int n_kv, const float* q_norm_w,
                                               const float* k_norm_w, float norm_eps, const float* cos_tab,
                                               const float* sin_tab, int pos, const int32_t* pos_dev,
                                               const ChattsKvCache* cache, size_t seq_stride, float* out, int n_splits,
                                               void* workspace, size_t workspace_bytes, chatts_stream_t stream) {
  return chatts::attention_decode_batched_impl(qkv_raw, batch, n_q, n_kv, q_norm_w, k_norm_w, norm_eps, cos_tab, sin_tab, pos,
                                               pos_dev, cache, seq_stride, out, nullptr, nullptr, n_splits, workspace,
                                               workspace_bytes, stream, nullptr);
}

extern "C" int chatts_attention_decode_fused(const float* qkv_raw, int n_q, int n_kv, const float* q_norm_w,
                                             const float* k_norm_w, float norm_eps, const float* cos_tab,
                                             const float* sin_tab, int pos, const int32_t* pos_dev,
                                             const ChattsKvCache* cache, float* out, int n_splits, void* workspace,
                                             size_t workspace_bytes, chatts_stream_t stream) {
  return chatts_attention_decode_batched(qkv_raw, 1, n_q, n_kv, q_norm_w, k_norm_w, norm_eps, cos_tab, sin_tab, pos, pos_dev,
                                         cache, 0, out, n_splits, workspace, workspace_bytes, stream);
}

