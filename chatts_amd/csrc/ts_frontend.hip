// ts_frontend.hip - sp-masked patchify of the padded [N, 2*Lmax] (value, mask) series tensor.
// Replaces the per-series Python loop of TimeSeriesEmbedding.forward
// (NetManAIOps/ChatTS chatts/vllm/chatts_vllm.py:93-183): there, 2 .item() host syncs and ~10 tiny
// torch ops per series; here one wave per series for the mask reduction and one wave per patch for
// the feature row, no host sync.
#include <type_traits>

#include "common.h"
#include "gemm_common.h"

namespace chatts {

// One wave per series: valid_len = sum(long(mask)) (chatts_vllm.py:98-99), patch_cnt = ceil(vl/ps).
// The (value, mask) pairs are read as float2 -> each lane streams 8 B, 512 B per wave instruction.  Eight of them are requested before the first is
// counted, at clamped addresses: a series is a chain of round trips otherwise, one per 64 steps (30 series of 1024: 10.0 us, now 6.1).
__device__ __forceinline__ void ts_count_series(const float* __restrict__ series, int i, int lmax, int patch, int lane, int32_t* vl_out, int64_t* pc_out) {
  const float2* row = reinterpret_cast<const float2*>(series) + (size_t)i * lmax;
  int cnt = 0;
  for (int t0 = lane; t0 < lmax; t0 += 64 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = row[t0 + u * 64 < lmax ? t0 + u * 64 : lmax - 1].y;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u * 64 < lmax) cnt += (int)(long long)v[u];      // .long(): truncate toward zero
  }
  cnt = wave_sum_i(cnt);
  if (lane == 0) {
    if (vl_out) vl_out[i] = cnt;
    if (pc_out) pc_out[i] = (int64_t)((cnt + patch - 1) / patch);
  }
}
__global__ __launch_bounds__(256) void ts_patch_cnt_kernel(const float* __restrict__ series, int n_series,
                                                          int lmax, int patch, int32_t* __restrict__ vl_out,
                                                          int64_t* __restrict__ pc_out) {
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave < n_series) ts_count_series(series, wave, lmax, patch, threadIdx.x & 63, vl_out, pc_out);
}

// Lengths that the host knows travel as kernel arguments: two copies from pageable memory took the device 5 us and the host 12 of an encoder call of 60.
// The counts from the masks, which the caller hands out, ride along.
constexpr int kTsByValue = 128;
struct TsLengths { int32_t len[kTsByValue], off[kTsByValue]; };
__global__ __launch_bounds__(256) void ts_lengths_kernel(TsLengths t, int count, int end, int32_t* __restrict__ valid_len, int32_t* __restrict__ row_off, const float* __restrict__ series,
                                                        int lmax, int patch, int64_t* __restrict__ patch_cnt) {
  const int tid = threadIdx.x, wave = (blockIdx.x * 256 + tid) >> 6;
  if (blockIdx.x == 0 && tid < count) {
    if (valid_len) valid_len[tid] = t.len[tid];
    row_off[tid] = t.off[tid];
    if (tid == count - 1) row_off[count] = end;
  }
  if (patch_cnt && wave < count) ts_count_series(series, wave, lmax, patch, tid & 63, nullptr, patch_cnt);
}

// Offsets of lengths that only the device knows: one wave, 64 series a turn.  It runs while the host waits for the lengths; sent behind that wait, as kernel arguments, the launch stood
// between the host and the first layer (2 us of a call of 90 to 150).
__global__ __launch_bounds__(64) void ts_offsets_kernel(const int32_t* __restrict__ valid_len, int n, int patch, int32_t* __restrict__ row_off) {
  const int lane = threadIdx.x;
  int before = 0;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int own = i0 + lane < n ? (valid_len[i0 + lane] + patch - 1) / patch : 0;
    int sum = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(sum, o, 64);
      if (lane >= o) sum += v;
    }
    if (i0 + lane < n) row_off[i0 + lane] = before + sum - own;
    before += __shfl(sum, 63, 64);
  }
  if (lane == 0) row_off[n] = before;
}

// One wave per output patch row.  Lanes 0..ps-1 own the ps values of the patch; in mode 1 every lane
// then copies position-embedding elements (ps*emb contiguous floats in the output row).
// The series owning patch row `p` is found by a binary search over row_off (N+1 ints, L2/L1 resident).
__global__ __launch_bounds__(256) void ts_patchify_kernel(ChattsPatchifyArgs a) {
  const int p = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (p >= a.total_patches) return;
  int lo = 0, hi = a.n_series;  // largest s with row_off[s] <= p
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.row_off[mid] <= p) lo = mid; else hi = mid;
  }
  const int s = lo;
  const int vl = a.valid_len[s];
  const int pp = p - a.row_off[s];          // patch index inside the series
  const int ps = a.patch_size;
  const float2* row = reinterpret_cast<const float2*>(a.series) + (size_t)s * a.lmax;
  // the row goes out as float32, or (out_hi / out_lo set) directly as the bf16 hi / lo planes of that float32 value - the
  // operand format of the first MLP GEMM (same split as chatts_split_bf16x2: hi = bf16(v), lo = bf16(v - hi))
  const size_t obase = (size_t)p * a.ld_out;
  auto put = [&](int col, float v) {
    if (a.out_hi) {
      uint16_t h, l;
      split_bf16x2(v, h, l);
      a.out_hi[obase + col] = h;
      a.out_lo[obase + col] = l;
    } else {
      a.out[obase + col] = v;
    }
  };
  const int t0 = pp * ps;
  const float last = row[vl - 1].x;          // last VALID value (chatts_vllm.py:122); vl >= 1 here
  int feat;
  if (a.mode == 1) {
    feat = ps + ps * a.emb_dim;
    if (lane < ps) {
      const int t = t0 + lane;
      put(lane, t < vl ? row[t].x : last);
    }
    // out[ps + j*emb + e] = pos_table[idx_j][e], idx_j = t0+j if valid else padding_idx (= max_seq_len)
    for (int q = lane; q < ps * a.emb_dim; q += 64) {
      const int j = q / a.emb_dim, e = q - j * a.emb_dim;
      const int t = t0 + j;
      const int idx = t < vl ? t : a.max_seq_len;
      put(ps + q, a.pos_table[(size_t)idx * a.emb_dim + e]);
    }
  } else if (a.mode == 2) {
    feat = 2 * ps;
    if (lane < ps) {
      const int t = t0 + lane;
      const int den = a.max_valid_len - 1 > 1 ? a.max_valid_len - 1 : 1;   // max(1, max_vl-1), :147
      put(2 * lane, t < vl ? row[t].x : last);
      put(2 * lane + 1, t < vl ? (float)t / (float)den : -1.0f);
    }
  } else {
    feat = ps;
    if (lane < ps) {
      const int t = t0 + lane;
      put(lane, t < vl ? row[t].x : last);
    }
  }
  for (int q = feat + lane; q < a.ld_out; q += 64) put(q, 0.f);   // K padding for the MFMA GEMM
}

// Value-preserved normalisation on the device (sp_encoding, chatts/utils/encoding_utils.py:23-37), one workgroup per series:
// mean, centred values, scale = max|x - mean| / 3 when some |x - mean| >= 3, and the (value, 1.0)-interleaved float32 rows
// of the padded encoder input - plus the statistics the prompt prefix prints.  Everything is float64 like the reference's
// numpy; the sum runs in a FIXED order (256 strided partial sums, then a binary tree), so it is reproducible, but it is not
// numpy's order: the mean can differ from np.mean in the last bit (max / min / ends are exact).
__global__ __launch_bounds__(256) void ts_normalise_kernel(const double* __restrict__ raw, const int32_t* __restrict__ len, int lmax,
                                                          float* __restrict__ enc, double* __restrict__ stats) {
  __shared__ double red[256];
  __shared__ double bc[2];
  const int s = blockIdx.x, tid = threadIdx.x;
  const int L = len[s];
  const double* x = raw + (size_t)s * lmax;
  float2* out = reinterpret_cast<float2*>(enc) + (size_t)s * lmax;
  double* st = stats + (size_t)s * 6;          // mean, factor, max, min, left, right
  if (L <= 0) {
    for (int t = tid; t < lmax; t += 256) out[t] = make_float2(0.f, 0.f);
    if (tid < 6) st[tid] = tid == 1 ? 1.0 : 0.0;
    return;
  }
  auto tree = [&](double v, int op) {            // op 0 sum, 1 max, 2 min; every thread returns the result
    red[tid] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if (tid < o) {
        const double a = red[tid], b = red[tid + o];
        red[tid] = op == 0 ? a + b : (op == 1 ? (a > b ? a : b) : (a < b ? a : b));
      }
      __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
  };
  double sum = 0.0, mx = -INFINITY, mn = INFINITY;
  for (int t = tid; t < L; t += 256) { const double v = x[t]; sum += v; mx = v > mx ? v : mx; mn = v < mn ? v : mn; }
  const double mean = tree(sum, 0) / (double)L;
  mx = tree(mx, 1);
  mn = tree(mn, 2);
  double dev = 0.0;
  for (int t = tid; t < L; t += 256) { const double d = fabs(x[t] - mean); dev = d > dev ? d : dev; }
  dev = tree(dev, 1);
  const double factor = dev >= 3.0 ? dev / 3.0 : 1.0;
  for (int t = tid; t < lmax; t += 256) {
    if (t < L) {
      double v = x[t] - mean;
      if (dev >= 3.0) v = v / factor;            // the reference divides in place (scaled /= factor), float64
      out[t] = make_float2((float)v, 1.0f);
    } else {
      out[t] = make_float2(0.f, 0.f);            // zero padding: mask 0 (encoding_utils.py:78-84)
    }
  }
  if (tid == 0) { st[0] = mean; st[1] = factor; st[2] = mx; st[3] = mn; st[4] = x[0]; st[5] = x[L - 1]; }
  (void)bc;
}

}  // namespace chatts

// ---- patchify + the first MLP layer in ONE launch --------------------------------------------------------------------------------------
// out0[p, n] = GELU(feat[p, :] . W0[n, :] + b0[n]) written as bf16 hi / lo planes - the operand of layer 1.  A wave owns 16 patch rows: it builds
// and splits their features in registers, straight from the series and the position table (the feature row never exists in memory), and walks over
// steps of 32 columns; W0 of a step comes to LDS once for the four waves of a workgroup, two steps ahead.  The MFMAs and their order are the prefill
// kernel's (per 32 K-values: lo pass, then hi pass; operands swapped, D = W . A^T): bit-identical planes.
// What bounds it: few patches - the chain offsets -> series -> MFMA -> store; many - vector operations, the 60 to 90 of an exact-erf GELU per output and the splits.
// It used to be a wave per 16 rows x 32 columns that built its features anew and read its W0 fragments (64-byte pieces of lines) from L2: 7.5 TB/s of
// those at many patches, and the features' loads one group after the other at few.  us before -> after: 1036 patches of 30 series, 5120 columns 64 -> 30
// (the loop over columns with W0 in registers alone: 39), 128 patches 14.6 -> 13.1, 16 patches, 4096 columns 10 -> 6.6.
namespace chatts {
// the 8 consecutive features k0 .. k0 + 7 (k0 = 32 s + 8 kc) of one patch row.  Every load is unconditional, at a clamped address (the tail value is row[vl - 1], a group
// past the features reads what another one reads), and selected afterwards: under a condition of the lane the compiler waits for each group before it
// asks for the next one, nine round trips in a row.  MODE is compile time.  Mode 1 needs patch size and embedding width multiples of 8 (every shipped
// config: 16 / 16): a group then lies wholly inside the value part or inside ONE position's embedding row, and with at most ten K-steps the
// value part lies inside the first (patch * (1 + emb) <= 320, emb >= 8).  emb8_inv = ceil(2^32 / (emb_dim / 8)), 0 for 1.
template <int MODE>
__device__ __forceinline__ void ts_feature8(const ChattsPatchifyArgs& a, unsigned emb8_inv, const float2* row, int vl, int t0, int s, int kc, float (&v)[8]) {
  const int ps = a.patch_size, k0 = s * 32 + kc * 8;
  if constexpr (MODE == 1) {
    const bool ok = k0 >= ps && k0 < ps + ps * a.emb_dim;
    const int q0 = ok ? k0 - ps : 0, j = emb8_inv ? (int)__umulhi((unsigned)q0 >> 3, emb8_inv) : q0 >> 3;
    const int t = t0 + j;
    const float* src = a.pos_table + (size_t)(t < vl ? t : a.max_seq_len) * a.emb_dim + (q0 - j * a.emb_dim);
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(src), x1 = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = ok ? (q < 4 ? x0[q & 3] : x1[q & 3]) : 0.f;      // (the value part: the caller's)
  } else if constexpr (MODE == 2) {      // (value, position) pairs: k even = value of t0 + k / 2, k odd = t / max(1, max_vl - 1) or -1
    const bool ok = k0 < 2 * ps;
    const int den = a.max_valid_len - 1 > 1 ? a.max_valid_len - 1 : 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int t = t0 + (ok ? (k0 >> 1) + q : 0);
      const float x = row[t < vl ? t : vl - 1].x;
      v[2 * q] = ok ? x : 0.f;
      v[2 * q + 1] = ok ? (t < vl ? (float)t / (float)den : -1.0f) : 0.f;
    }
  } else {
    const bool ok = k0 < ps;
#pragma unroll
    for (int q = 0; q < 8; ++q) { const int t = t0 + (ok ? k0 + q : 0); const float x = row[t < vl ? t : vl - 1].x; v[q] = ok ? x : 0.f; }
  }
}

constexpr int kL0Waves = 4, kL0Cols = 32;      // waves (16 rows each) of a workgroup, columns of a step

// Lengths that the host knows, for the first layer itself: no launch before it writes them and no wave waits for them (2.3 us of device and 4 of host time a call).  Up to kL0Known series;
// places behind the last one hold offsets that no row reaches.
constexpr int kL0Known = 64;
struct TsKnown {
  int32_t off[kL0Known], len[kL0Known];
  int32_t n;
  int64_t* patch_cnt;      // counts from the masks, by workgroups of their own (the last of grid.y), or NULL
};

struct TsOnDevice {        // row_off and valid_len (an instance of its own: one that takes either is 0.8 us of 28 slower for them)
  static constexpr int32_t n = 0;
};

template <int KSTEPS, int MODE, typename LENGTHS>      // K-steps of 32 (feature count rounded up) and the feature mode: compiled in, so that every load is in flight at once
__global__ __launch_bounds__(64 * kL0Waves, 3) void ts_layer0_kernel(ChattsPatchifyArgs a, unsigned emb8_inv, const uint16_t* w0, int ldw, const float* b0, int hidden, int steps_each,
                                                                     uint16_t* out_hi, uint16_t* out_lo, int ld_out, int tiled, LENGTHS known) {
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  constexpr bool KNOWN = std::is_same<LENGTHS, TsKnown>::value;
  // W0 of a step: 32 rows of 4 KSTEPS 16-byte chunks, twice.  Chunk c of a K-step of row r lies at place c ^ (r >> turn): eight rows' chunks then meet
  // different banks whatever KSTEPS makes of the row's length
  constexpr int ROW = 4 * KSTEPS, PIECES = 2 * KSTEPS, TURN = KSTEPS % 2 ? 2 : (KSTEPS % 4 ? 1 : 0);
  __shared__ __attribute__((aligned(1024))) char smem[2][PIECES * 1024];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = ((int)blockIdx.y * kL0Waves + wave) * 16;
  if (KNOWN && (int)blockIdx.y * kL0Waves * 16 >= a.total_patches) {      // (a whole workgroup)
    if constexpr (KNOWN)
      for (int i = (int)blockIdx.x * kL0Waves + wave; i < known.n; i += (int)gridDim.x * kL0Waves) ts_count_series(a.series, i, a.lmax, a.patch_size, lane, nullptr, known.patch_cnt);
    return;
  }
  const bool mine = r0 < a.total_patches;                      // (else a wave that only fetches W0)
  const int frow = lane & 15, kc = lane >> 4;                  // this lane's row of a 16-row block, and its 8 K-values of a 32-deep step
  int n0 = (int)blockIdx.x * steps_each * kL0Cols;
  const int n_end = n0 + steps_each * kL0Cols < hidden ? n0 + steps_each * kL0Cols : hidden;
  auto fetch = [&](int n, int b) __attribute__((always_inline)) {        // (rows past the end of W0 repeat its last one; their sums are dropped)
#pragma unroll
    for (int q = 0; q < (PIECES + kL0Waves - 1) / kL0Waves; ++q) {
      const int piece = q * kL0Waves + wave;
      if (q * kL0Waves + kL0Waves > PIECES && piece >= PIECES) continue;
      const int c = piece * 64 + lane, r = c / ROW, x = c - r * ROW;
      const int row = n + r < hidden ? n + r : hidden - 1;
      __builtin_amdgcn_global_load_lds((gptr_t)(w0 + (size_t)row * ldw + ((x & ~3) | ((x & 3) ^ ((r >> TURN) & 3))) * 8), (lptr_t)(smem[b] + piece * 1024), 16, 0, 0);
    }
  };
  // the patch row this lane feeds, clamped to the last real row (stores are masked).  Its series: of lengths by value, the last that begins at or before the row (scalar
  // loads, 16 series at a time); up to 63 series - lane i holds
  // row_off[i] / valid_len[i] (ONE round trip), the search is a wave-uniform walk over lanes and two ds_bpermute; more series - the
  // binary search of ts_patchify_kernel (log2 N dependent round trips)
  const int nser = a.n_series;
  int p = r0 + frow;
  if (p > a.total_patches - 1) p = a.total_patches - 1;
  const int my_off = KNOWN ? 0 : a.row_off[lane <= nser ? lane : nser];      // (requested before the branch)
  const int my_vl = KNOWN ? 0 : a.valid_len[lane < nser ? lane : nser - 1];
  int sidx = 0, off = 0, vl = 0;
  if constexpr (KNOWN) {
    for (int i0 = 0; i0 < known.n; i0 += 16)
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int o = known.off[i0 + u], l = known.len[i0 + u];
        const bool at = o <= p;
        sidx = at ? i0 + u : sidx;
        off = at ? o : off;
        vl = at ? l : vl;
      }
  } else if (nser <= 63) {
    for (int i = 1; i < nser; ++i) sidx += __builtin_amdgcn_readlane(my_off, i) <= p ? 1 : 0;
    off = __shfl(my_off, sidx, 64);
    vl = __shfl(my_vl, sidx, 64);
  } else {
    int lo = 0, hi = nser;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (a.row_off[mid] <= p) lo = mid; else hi = mid;
    }
    sidx = lo;
    off = a.row_off[lo];
    vl = a.valid_len[lo];
  }
  const int t0 = (p - off) * a.patch_size;
  const float2* rowp = reinterpret_cast<const float2*>(a.series) + (size_t)sidx * a.lmax;
  // every feature load of the block before the first use, and the first two steps of W0 behind them
  float raw[KSTEPS][8];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) ts_feature8<MODE>(a, emb8_inv, rowp, vl, t0, s, kc, raw[s]);
  float val[8];
  if constexpr (MODE == 1) {
#pragma unroll
    for (int q = 0; q < 8; ++q) { const int t = t0 + kc * 8 + q; val[q] = rowp[t < vl ? t : vl - 1].x; }
  }
  fetch(n0, 0);
  if (n0 + kL0Cols < n_end) fetch(n0 + kL0Cols, 1);
  if constexpr (MODE == 1) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      asm volatile("" : "+v"(val[q]));                         // (keeps the loads out of the condition)
      if (kc * 8 < a.patch_size) raw[0][q] = val[q];
    }
  }
  bf16x8_t ahi[KSTEPS], alo[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const __bf16 h = (__bf16)raw[s][q];
      ahi[s][q] = h;
      alo[s][q] = (__bf16)(raw[s][q] - (float)h);
    }
  const int tok = r0 + frow;
  const bool live = tok < a.total_patches;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  for (int b = 0; n0 < n_end; n0 += kL0Cols, b ^= 1) {
    // lane holds D[feature n0 + 16 j + 4 kc + r][token r0 + frow]: bias, exact-erf GELU, split, 8-byte stores (ring_store's arithmetic)
    bf16x4_t hv[2], lv[2];
    if (mine) {
      f32x4 bias[2], acc[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int fb = n0 + j * 16 + kc * 4;
        bias[j] = b0 ? *reinterpret_cast<const f32x4*>(b0 + (fb < hidden ? fb : 0)) : (f32x4){0.f, 0.f, 0.f, 0.f};
        acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
      const char* w = smem[b] + (frow * ROW + (kc ^ ((frow >> TURN) & 3))) * 16;      // (16 rows on: the same place, 16 >> TURN is a multiple of 4)
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        bf16x8_t wf[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) wf[j] = *reinterpret_cast<const bf16x8_t*>(w + j * 16 * ROW * 16 + s * 64);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], alo[s], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], ahi[s], acc[j], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma clang fp contract(off)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = gelu_erf_f(acc[j][r] + bias[j][r]);
          const __bf16 h = (__bf16)v;
          hv[j][r] = h;
          lv[j][r] = (__bf16)(v - (float)h);
        }
      }
    }
    // what is waited for: the next step's pieces of this wave, and the stores of the step before; then all waves are through with this step's W0 and have the next one's
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (live)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int fb = n0 + j * 16 + kc * 4;
        if (fb < hidden) {
          const size_t at = plane_at(tok, fb, ld_out, tiled);
          *reinterpret_cast<bf16x4_t*>(out_hi + at) = hv[j];
          *reinterpret_cast<bf16x4_t*>(out_lo + at) = lv[j];
        }
      }
    if (n0 + 2 * kL0Cols < n_end) fetch(n0 + 2 * kL0Cols, b);
  }
}
}  // namespace chatts

using namespace chatts;

extern "C" int chatts_ts_normalise(const double* raw, const int32_t* lengths, int n_series, int lmax, float* enc, double* stats,
                                   chatts_stream_t stream) {
  CHATTS_REQUIRE(n_series >= 0 && lmax >= 0, CHATTS_E_BADARG, "ts_normalise: bad sizes n=%d lmax=%d", n_series, lmax);
  if (n_series == 0 || lmax == 0) return CHATTS_OK;
  CHATTS_REQUIRE(raw && lengths && enc && stats, CHATTS_E_BADARG, "ts_normalise: null pointer");
  hipLaunchKernelGGL(ts_normalise_kernel, dim3(n_series), dim3(256), 0, as_stream(stream), raw, lengths, lmax, enc, stats);
  CHATTS_CHECK_LAUNCH("ts_normalise");
  return CHATTS_OK;
}

extern "C" int chatts_ts_patch_cnt(const float* series, int n_series, int lmax, int patch_size,
                                   int32_t* valid_len, int64_t* patch_cnt, chatts_stream_t stream) {
  CHATTS_REQUIRE(n_series >= 0 && lmax >= 0 && patch_size > 0, CHATTS_E_BADARG,
                 "ts_patch_cnt: bad sizes n=%d lmax=%d patch=%d", n_series, lmax, patch_size);
  if (n_series == 0) return CHATTS_OK;
  CHATTS_REQUIRE(series != nullptr || lmax == 0, CHATTS_E_BADARG, "ts_patch_cnt: null series");
  CHATTS_REQUIRE(valid_len || patch_cnt, CHATTS_E_BADARG, "ts_patch_cnt: no output");
  const int blocks = (n_series + 3) / 4;
  hipLaunchKernelGGL(ts_patch_cnt_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), series, n_series,
                     lmax, patch_size, valid_len, patch_cnt);
  CHATTS_CHECK_LAUNCH("ts_patch_cnt");
  return CHATTS_OK;
}

extern "C" int chatts_ts_lengths(const int32_t* lengths, int n_series, int patch_size, int32_t* valid_len, int32_t* row_off, const float* series, int lmax, int64_t* patch_cnt,
                                 chatts_stream_t stream) {
  CHATTS_REQUIRE(n_series >= 0 && lmax >= 0 && patch_size > 0, CHATTS_E_BADARG, "ts_lengths: bad sizes n=%d lmax=%d patch=%d", n_series, lmax, patch_size);
  if (n_series == 0) return CHATTS_OK;
  if (!lengths) {
    CHATTS_REQUIRE(valid_len && row_off && !patch_cnt, CHATTS_E_BADARG, "ts_lengths: lengths on the device need valid_len and row_off, without counts");
    hipLaunchKernelGGL(ts_offsets_kernel, dim3(1), dim3(64), 0, as_stream(stream), valid_len, n_series, patch_size, row_off);
    CHATTS_CHECK_LAUNCH("ts_offsets");
    return CHATTS_OK;
  }
  CHATTS_REQUIRE(row_off && (!patch_cnt || series || lmax == 0), CHATTS_E_BADARG, "ts_lengths: null pointer");
  int at = 0;
  for (int i0 = 0; i0 < n_series; i0 += kTsByValue) {
    const int count = n_series - i0 < kTsByValue ? n_series - i0 : kTsByValue;
    TsLengths t{};
    for (int i = 0; i < count; ++i) {
      CHATTS_REQUIRE(lengths[i0 + i] >= 0, CHATTS_E_BADARG, "ts_lengths: series %d of %d steps", i0 + i, lengths[i0 + i]);
      t.len[i] = lengths[i0 + i];
      t.off[i] = at;
      at += (lengths[i0 + i] + patch_size - 1) / patch_size;
    }
    hipLaunchKernelGGL(ts_lengths_kernel, dim3(patch_cnt ? (count + 3) / 4 : 1), dim3(256), 0, as_stream(stream), t, count, at, valid_len ? valid_len + i0 : nullptr, row_off + i0,
                       series ? series + (size_t)i0 * lmax * 2 : nullptr, lmax, patch_size, patch_cnt ? patch_cnt + i0 : nullptr);
    CHATTS_CHECK_LAUNCH("ts_lengths");
  }
  return CHATTS_OK;
}

extern "C" int chatts_ts_patchify(const ChattsPatchifyArgs* a, chatts_stream_t stream) {
  CHATTS_REQUIRE(a != nullptr, CHATTS_E_BADARG, "ts_patchify: null args");
  CHATTS_REQUIRE(a->total_patches >= 0 && a->n_series >= 0, CHATTS_E_BADARG, "ts_patchify: negative size");
  if (a->total_patches == 0) return CHATTS_OK;
  CHATTS_REQUIRE(a->series && a->row_off && a->valid_len && (a->out || (a->out_hi && a->out_lo)), CHATTS_E_BADARG,
                 "ts_patchify: null pointer");
  CHATTS_REQUIRE(a->patch_size > 0 && a->patch_size <= 64, CHATTS_E_SHAPE, "ts_patchify: patch_size %d not in 1..64",
                 a->patch_size);
  CHATTS_REQUIRE(a->mode >= 0 && a->mode <= 2, CHATTS_E_BADARG, "ts_patchify: mode %d", a->mode);
  const int feat = a->mode == 1 ? a->patch_size * (1 + a->emb_dim) : (a->mode == 2 ? 2 * a->patch_size : a->patch_size);
  CHATTS_REQUIRE(a->ld_out >= feat, CHATTS_E_SHAPE, "ts_patchify: ld_out %d < features %d", a->ld_out, feat);
  if (a->mode == 1)
    CHATTS_REQUIRE(a->pos_table && a->emb_dim > 0 && a->max_seq_len > 0, CHATTS_E_BADARG,
                   "ts_patchify: position table missing");
  const int blocks = (a->total_patches + 3) / 4;
  hipLaunchKernelGGL(ts_patchify_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), *a);
  CHATTS_CHECK_LAUNCH("ts_patchify");
  return CHATTS_OK;
}

// Whole encoder in one call (the C-ABI SURVEY.md section 8b proposes for a3 + a4): patchify, then the MLP
// (Linear + exact-erf GELU) x (n-1) + Linear, ping-ponging between two caller-owned [P, H] buffers.
// lengths: the same on the host, or NULL.  Then row_off and valid_len are written by chatts_ts_lengths where the first layer does not take them as arguments, and patch_cnt by one of the two.
static int ts_encode(const float* series, const int32_t* lengths, int32_t* row_off, int32_t* valid_len, int64_t* patch_cnt, int n_series, int lmax,
                     int max_valid_len, int total_patches, const ChattsTsWeights* w, const chatts_bf16* const* w_tiled, float* feat, float* h0,
                     float* h1, float* out, void* workspace, size_t workspace_bytes, chatts_stream_t stream) {
  CHATTS_REQUIRE(w != nullptr && w->num_layers >= 1 && w->num_layers <= 8, CHATTS_E_BADARG, "ts_encode: bad weights");
  if (total_patches == 0) return CHATTS_OK;
  StageRange stage("chatts.ts_encode");
  CHATTS_REQUIRE(feat && out && (w->num_layers < 2 || h0) && (w->num_layers < 3 || h1), CHATTS_E_BADARG,
                 "ts_encode: null buffer");
  ChattsPatchifyArgs pa{};
  pa.series = series; pa.row_off = row_off; pa.valid_len = valid_len; pa.pos_table = w->pos_table; pa.out = feat;
  pa.n_series = n_series; pa.lmax = lmax; pa.patch_size = w->patch_size; pa.mode = w->mode; pa.emb_dim = w->emb_dim;
  pa.max_seq_len = w->max_seq_len; pa.max_valid_len = max_valid_len; pa.total_patches = total_patches;
  pa.ld_out = w->in_features_pad;
  // Plane path (P > 1 and every K a multiple of 64): each activation matrix lives as bf16 hi / lo planes inside the caller's
  // float32 scratch of the same byte size (4 B per element = 2 + 2) - patchify writes the planes of layer 0's operand, every
  // GELU epilogue writes the planes of the next layer's, and the GEMMs stage all operands with whole-line LDS-DMA
  // (gemm_stream_kernel for few rows: the 213 MB of MLP weights are streamed once; gemm_ring_kernel above).  The values are
  // the splits of exactly the float32 numbers the float32 path would hold, so both paths give the same result.
  const int P = total_patches, H = w->hidden;
  const bool planes = P > 1 && w->in_features_pad % 64 == 0 && H % 64 == 0 && opt_get(OPT_TS_F32_PATH, 0) == 0;
  // The prefill kernel from 65 rows on, where the weights lie in its blocks and stream_leaves_cus; else, up to 128 rows, the weight stream.  Activations between its layers in blocks, too.
  const bool mid = planes && w_tiled && P > 64 && P <= 128 && stream_leaves_cus(P, H, H);
  const bool tile = planes && (mid ? opt_get(OPT_PLANE_TILES, 1) != 0 : planes_tiled_for(P, H, H));
  // The weights in blocks likewise, where the caller has them so: a 1 KB piece of the loader is 1 KB of memory.  1036 rows of 5120 x 5120, us a layer: 88.6 -> 82.4.
  auto hi_of = [&](float* buf) { return reinterpret_cast<chatts_bf16*>(buf); };
  auto lo_of = [&](float* buf, int k) { return reinterpret_cast<chatts_bf16*>(buf) + (size_t)P * k; };
  if (planes) { pa.out = nullptr; pa.out_hi = hi_of(feat); pa.out_lo = lo_of(feat, w->in_features_pad); }
  int rc;
  float* cur = feat;
  int k = w->in_features_pad;
  int l0 = 0;
  // patchify + layer 0 as one launch (ts_layer0_kernel) when layer 0 is a hidden layer of the plane path: its GELU output goes out as the
  // planes layer 1 reads; the feature matrix is never written.  TS_L0_FUSED=0 keeps the two-launch form (bit-identical).
  const int feat_n = w->mode == 1 ? w->patch_size * (1 + w->emb_dim) : (w->mode == 2 ? 2 * w->patch_size : w->patch_size);
  const int ksteps = (feat_n + 31) / 32;
  const bool l0_shape = w->mode == 1 ? (w->patch_size % 8 == 0 && w->emb_dim % 8 == 0 && ksteps <= 10) : (w->patch_size % 8 == 0 && ksteps <= 2);
  const bool fused = planes && w->num_layers >= 2 && H % 16 == 0 && ksteps >= 1 && l0_shape && ksteps * 32 <= w->in_features_pad && h0 &&
      ((uintptr_t)w->w[0] % 16) == 0 && ((uintptr_t)w->b[0] % 16) == 0 && ((uintptr_t)w->pos_table % 16) == 0 && opt_get(OPT_TS_L0_FUSED, 1) != 0;
  TsKnown known{};
  if (lengths) {
    if (fused && n_series <= kL0Known && series) {
      known.n = n_series; known.patch_cnt = patch_cnt;
      for (int i = 0, at = 0; i < kL0Known; ++i) {
        known.off[i] = i < n_series ? at : 0x7fffffff;
        if (i < n_series) { known.len[i] = lengths[i]; at += (lengths[i] + w->patch_size - 1) / w->patch_size; }
      }
    } else if ((rc = chatts_ts_lengths(lengths, n_series, w->patch_size, valid_len, row_off, series, lmax, patch_cnt, stream)) != 0) {
      return rc;
    }
  }
  if (fused) {
    CHATTS_REQUIRE(pa.series && pa.row_off && pa.valid_len && (w->mode != 1 || (pa.pos_table && w->emb_dim > 0 && w->max_seq_len > 0)), CHATTS_E_BADARG,
                   "ts_encode: null series / offsets / position table");
    // four row blocks a workgroup; the columns in as many parts as three workgroups per CU ask for
    const int groups = (P + 16 * kL0Waves - 1) / (16 * kL0Waves), steps = (H + kL0Cols - 1) / kL0Cols;
    int parts = 3 * device_cus() / groups;
    parts = parts < 1 ? 1 : (parts > steps ? steps : parts);
    const int steps_each = (steps + parts - 1) / parts, emb8 = w->mode == 1 ? w->emb_dim / 8 : 1;
    const unsigned emb8_inv = emb8 > 1 ? (unsigned)((0x100000000ull + emb8 - 1) / emb8) : 0u;      // (exact for the at most 40 groups of a row)
    const dim3 grid((steps + steps_each - 1) / steps_each, groups + (known.n && known.patch_cnt ? 1 : 0)), block(64 * kL0Waves);
    uint16_t* oh = hi_of(h0);
    uint16_t* ol = lo_of(h0, H);
#define CHATTS_TS_L0_OF(KS, MD, L, known) hipLaunchKernelGGL((ts_layer0_kernel<KS, MD, L>), grid, block, 0, as_stream(stream), pa, emb8_inv, w->w[0], w->in_features_pad, w->b[0], H, steps_each, oh, ol, H, tile ? P & ~15 : 0, known)
#define CHATTS_TS_L0(KS, MD) if (known.n) CHATTS_TS_L0_OF(KS, MD, TsKnown, known); else CHATTS_TS_L0_OF(KS, MD, TsOnDevice, TsOnDevice{})
    if (w->mode == 1) {
      switch (ksteps) {
        case 1: CHATTS_TS_L0(1, 1); break;
        case 2: CHATTS_TS_L0(2, 1); break;
        case 3: CHATTS_TS_L0(3, 1); break;
        case 4: CHATTS_TS_L0(4, 1); break;
        case 5: CHATTS_TS_L0(5, 1); break;
        case 6: CHATTS_TS_L0(6, 1); break;
        case 7: CHATTS_TS_L0(7, 1); break;
        case 8: CHATTS_TS_L0(8, 1); break;
        case 9: CHATTS_TS_L0(9, 1); break;
        default: CHATTS_TS_L0(10, 1); break;
      }
    } else if (w->mode == 2) {
      if (ksteps == 1) { CHATTS_TS_L0(1, 2); } else { CHATTS_TS_L0(2, 2); }
    } else {
      if (ksteps == 1) { CHATTS_TS_L0(1, 0); } else { CHATTS_TS_L0(2, 0); }
    }
#undef CHATTS_TS_L0
#undef CHATTS_TS_L0_OF
    CHATTS_CHECK_LAUNCH("ts_layer0");
    cur = h0;
    k = H;
    l0 = 1;
  } else {
    if ((rc = chatts_ts_patchify(&pa, stream)) != 0) return rc;
  }
  for (int l = l0; l < w->num_layers; ++l) {
    const bool last = l == w->num_layers - 1;
    float* dst = last ? out : ((l & 1) ? h1 : h0);
    ChattsLinearArgs la{};
    la.w = w->w[l]; la.bias = w->b[l]; la.m = P; la.n = H; la.k = k;
    la.lda = k; la.ldw = k; la.ldc = H; la.epilogue = last ? CHATTS_EPI_NONE : CHATTS_EPI_GELU;
    la.workspace = workspace; la.workspace_bytes = workspace_bytes;
    if ((tile || mid) && w_tiled && l > 0) la.w_tiled = w_tiled[l];
    if (planes) {
      la.a_hi = hi_of(cur); la.a_lo = lo_of(cur, k); la.ld_planes = k;
      if (last) la.c = dst;
      else { la.c_hi = hi_of(dst); la.c_lo = lo_of(dst, H); la.ld_cplanes = H; }
    } else {
      la.a = cur; la.c = dst;
    }
    if ((rc = linear_tiled(&la, stream, {tile && l > 0, tile && !last, false, mid && l > 0})) != 0) return rc;
    cur = dst;
    k = H;
  }
  return CHATTS_OK;
}
extern "C" int chatts_ts_encode_tiled(const float* series, const int32_t* row_off, const int32_t* valid_len, int n_series, int lmax,
                                int max_valid_len, int total_patches, const ChattsTsWeights* w, const chatts_bf16* const* w_tiled, float* feat, float* h0,
                                float* h1, float* out, void* workspace, size_t workspace_bytes, chatts_stream_t stream) {
  return ts_encode(series, nullptr, const_cast<int32_t*>(row_off), const_cast<int32_t*>(valid_len), nullptr, n_series, lmax, max_valid_len, total_patches, w, w_tiled, feat, h0, h1, out,
                   workspace, workspace_bytes, stream);
}
extern "C" int chatts_ts_encode_known(const float* series, const int32_t* lengths, int n_series, int lmax, int32_t* valid_len, int32_t* row_off, int64_t* patch_cnt, const ChattsTsWeights* w,
                                      const chatts_bf16* const* w_tiled, float* feat, float* h0, float* h1, float* out, void* workspace, size_t workspace_bytes, chatts_stream_t stream) {
  CHATTS_REQUIRE(w && lengths && valid_len && row_off && n_series >= 0 && lmax >= 0 && w->patch_size > 0, CHATTS_E_BADARG, "ts_encode_known: bad arguments");
  int total = 0, longest = 0;
  for (int i = 0; i < n_series; ++i) {
    CHATTS_REQUIRE(lengths[i] >= 0 && lengths[i] <= lmax, CHATTS_E_BADARG, "ts_encode_known: series %d of %d steps in rows of %d", i, lengths[i], lmax);
    total += (lengths[i] + w->patch_size - 1) / w->patch_size;
    if (lengths[i] > longest) longest = lengths[i];
  }
  if (total == 0) return chatts_ts_lengths(lengths, n_series, w->patch_size, valid_len, row_off, series, lmax, patch_cnt, stream);
  return ts_encode(series, lengths, row_off, valid_len, patch_cnt, n_series, lmax, longest, total, w, w_tiled, feat, h0, h1, out, workspace, workspace_bytes, stream);
}
extern "C" int chatts_ts_encode(const float* series, const int32_t* row_off, const int32_t* valid_len, int n_series, int lmax, int max_valid_len, int total_patches, const ChattsTsWeights* w,
                                float* feat, float* h0, float* h1, float* out, void* workspace, size_t workspace_bytes, chatts_stream_t stream) {
  return chatts_ts_encode_tiled(series, row_off, valid_len, n_series, lmax, max_valid_len, total_patches, w, nullptr, feat, h0, h1, out, workspace, workspace_bytes, stream);
}

