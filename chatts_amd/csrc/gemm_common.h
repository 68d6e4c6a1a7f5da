// gemm_common.h - what the MFMA GEMM kernels share: the launch parameters and the small epilogue helpers (gemm.hip, gemm_ring.hip).
#pragma once
#include "common.h"

namespace chatts {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct GemmParams {
  const float* a;
  const uint16_t* w;
  const float* bias;
  const float* resid;
  float* c;          // final output, or split-K partials [sk][M][N]
  int m, n, k, lda, ldw, ldc, epilogue;
  int k_per_split;   // multiple of 32
  int direct;        // 1: apply epilogue here; 0: write raw partials
  const uint8_t* w8;     // optional fp8 (e4m3fn) copy of W: streamed instead of the bf16 copy, widened (exactly) to
  const float* w8_scale; // bf16 while it is staged to LDS; the per-row power-of-two scale is applied in the epilogue
  int ldw8;
  int w8_format;         // CHATTS_W8_FP8 / CHATTS_W8_INT8 (gemm_stream_kernel only; the other kernels never see an int8 copy)
  uint16_t* c_hi;        // optional: the output goes out as bf16 hi / lo planes [M, ldcp] (the next GEMM's operand
  uint16_t* c_lo;        // format) instead of float32 c
  int ldcp;
  const uint16_t* wt;    // optional (gemm_ring_kernel): W in the tiled layout of chatts_tile_bf16 - a 1 KB LDS-DMA piece is 1 KB of memory
  int planes_tiled;      // a_hi / a_lo are in that layout too
  int a_tiled, c_tiled;  // ... or their first so many rows are (plane_at), and those of c_hi / c_lo
  float glu_limit, glu_alpha;
  int64_t a_stride, w_stride, c_stride;   // several products of one shape (gemm_stream_kernel, grid y)
  // RMSNorm split over two projections of few rows (gemm_rows.hip): the row factor 1 / rms comes from the producer's partial sums of squares
  const float* row_ss;   // [16][256], or NULL
  int row_ss_parts;
  float row_eps;
  const float* post_w;   // with post_ss: planes of post_w * c beside c, and the sums of squares of this launch's columns
  float* post_ss;
  uint16_t* post_hi;
  uint16_t* post_lo;
  int ld_post;
};

__device__ __forceinline__ void store_planes(uint16_t* hi, uint16_t* lo, size_t off, float v) {
  // no contraction: when v is a product (SwiGLU) the compiler would otherwise fold it into the subtraction as an FMA and
  // lo would no longer be the split of the ROUNDED float32 value the float32 path stores
#pragma clang fp contract(off)
  const __bf16 h = (__bf16)v;
  const __bf16 l = (__bf16)(v - (float)h);
  hi[off] = __builtin_bit_cast(uint16_t, h);
  lo[off] = __builtin_bit_cast(uint16_t, l);
}

__device__ __forceinline__ void store_planes4(uint16_t* hi, uint16_t* lo, f32x4 v) {      // the same for four neighbours, 8 bytes a store
#pragma clang fp contract(off)
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  bf16x4_t hv, lv;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const __bf16 h = (__bf16)v[j];
    hv[j] = h;
    lv[j] = (__bf16)(v[j] - (float)h);
  }
  *reinterpret_cast<bf16x4_t*>(hi) = hv;
  *reinterpret_cast<bf16x4_t*>(lo) = lv;
}

// eight 8-bit weights as bf16, exactly: two a instruction (by way of float32 it took two for that, and they are most of what a few-rows kernel issues).
__device__ __forceinline__ bf16x8_t widen_fp8(u32x2 q8) {
  bf16x8_t bv = {};
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(q8[i], 1.f, false), hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(q8[i], 1.f, true);
    bv[4 * i] = lo[0]; bv[4 * i + 1] = lo[1]; bv[4 * i + 2] = hi[0]; bv[4 * i + 3] = hi[1];
  }
#endif
  return bv;
}
__device__ __forceinline__ bf16x8_t widen_i8(u32x2 q8) {
  const int a0 = (int)q8.x, a1 = (int)q8.y;
  bf16x8_t bv;
  bv[0] = (__bf16)(float)((a0 << 24) >> 24); bv[1] = (__bf16)(float)((a0 << 16) >> 24);
  bv[2] = (__bf16)(float)((a0 << 8) >> 24);  bv[3] = (__bf16)(float)(a0 >> 24);
  bv[4] = (__bf16)(float)((a1 << 24) >> 24); bv[5] = (__bf16)(float)((a1 << 16) >> 24);
  bv[6] = (__bf16)(float)((a1 << 8) >> 24);  bv[7] = (__bf16)(float)(a1 >> 24);
  return bv;
}

__device__ __forceinline__ float gelu_erf_f(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f)); }
__device__ __forceinline__ float relu2_f(float x) { const float r = fmaxf(x, 0.f); return r * r; }      // the square of relu
__device__ __forceinline__ float silu_g(float x) { return x / (1.0f + expf(-x)); }

__device__ __forceinline__ float glu_value(int epilogue, float g, float u, float limit, float alpha) {
  return epilogue == CHATTS_EPI_SWIGLU ? silu_g(g) * u : (epilogue == CHATTS_EPI_GEGLU ? gelu_tanh_glu(g, u) : clamp_glu(g, u, limit, alpha));
}

// Which planes of a projection lie as plane_at has them, whole blocks of 16 rows in tiles: A, the result's, those of the norm behind it.  Only for calls that take gemm_ring_kernel:
// planes_tiled_for says which do.  The loader then reads 1 KB at a time instead of 16 half lines that lie a row apart on the same channels of L2: us row-major / in tiles, W in
// tiles both times: 223 rows 24576 x 4096 gated 95.0 / 82.7, 6144 x 4096 35.9 / 32.0, 5120 x 5120 39.1 / 34.1; 798 rows 7168 x 5120 108 / 99, 27648 x 5120 gated 358 / 344, 5120 x 5120
// 83.2 / 81.8; 1473 rows 7168 x 5120 211 / 185, 4096 x 12288 242 / 229.  The same products in the same order: the same bits.
struct PlaneTiles {
  bool a, c, post;
  bool ring = false;      // the prefill kernel whatever the form of the planes
};
// 17 .. 95 rows on planes from this K on (up to 64 rows, and up to 128 where N is 8192 at most, the weight stream runs; else the prefill kernel): the register-staged kernel, which takes
// float32, needs 1.2 to 1.6 times as long.  us with the epilogue, float32 / planes: 17 rows 6144 x 4096 19.7 / 13.9, 24576 x 4096 gated 51.5 / 42.4, 4096 x 12288 34.2 / 21.7, 2048 x 2048
// 11.2 / 8.0; 48 rows 7168 x 5120 30.2 / 22.6, 27648 x 5120 gated 85.9 / 64.1; 80 rows 5120 x 13824 57.0 / 44.1, 8192 x 2048 23.7 / 20.5.  Shorter K is not the weight stream's.
constexpr int kMidPlanesK = 1024;
bool planes_tiled_for(int m, int n, int k);      // (gemm.hip: of the A of an m x n x k product)
bool stream_leaves_cus(int m, int n, int k);     // (gemm.hip: 65 .. 128 rows with W in tiles are the prefill kernel's)
// The sums that a projection of few rows left in the workspace, [sk][rows][n], for a reader that adds them up itself (sk == 0: none were left, c is written).  A launch of a captured graph
// takes 1.7 us before it does anything, and the sums' own launch does 0.3 us of work on 16 rows.
// Where the line lies: splits are left wherever a reader takes them, as no measured cell lost.  Attention: see attn_takes_splits.  Mixed layers, steps of eight layers with the same tokens on
// every route, us with all sums in launches of their own / those of the mixers left / those of the norm, too: width 2048, 9, 10, 12, 16 rows 810 / 788 / 772, 829 / 804 / 789, 858 / 831 / 816,
// 893 / 868 / 854 (runs of one route differ by 1 to 4); width 4096, 9 to 16 rows 0 to 6 us for the mixers and 3 to 24 for the norm (of 1900 to 2190; runs differ by 5 to 20); 8 rows and
// fewer take kernels without splits.  More than eight (mixers, attention) or sixteen (norm) splits keep their launch: a reader asks for all of them at once, in registers.
constexpr int kMostSplitSums = 8, kMostNormSums = 16;      // splits that a reader takes, and those of a norm
struct SplitSums {
  const float* slabs = nullptr;
  const float *scale = nullptr, *bias = nullptr;      // per column, or NULL
  size_t plane = 0;         // floats of a split
  int sk = 0, n = 0;
  int most = kMostSplitSums;      // asked for: splits that may be left
};
// four neighbours, in splitk_epilogue_v4_kernel's order: the same bits
template <int S>
__device__ __forceinline__ f32x4 split_sum4(const SplitSums& p, int row, int col) {
  const float* at = p.slabs + (size_t)row * p.n + col;
  f32x4 t[S], f, b, v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S; ++s) t[s] = *reinterpret_cast<const f32x4*>(at + (s < p.sk ? s : p.sk - 1) * p.plane);
  if (p.scale) f = *reinterpret_cast<const f32x4*>(p.scale + col);
  if (p.bias) b = *reinterpret_cast<const f32x4*>(p.bias + col);
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < p.sk) v += t[s];
  if (p.scale) v *= f;
  if (p.bias) v += b;
  return v;
}
int linear_tiled(const ChattsLinearArgs* a, chatts_stream_t stream, PlaneTiles tiles, SplitSums* leave = nullptr);      // chatts_linear on such planes (decoder.hip)
int gru_decode(const ChattsGruArgs* a, const SplitSums& in, hipStream_t s);      // chatts_gru_decode on what a projection left (gru.hip)
// what attention and a selective scan that read one projection do before their own launches, one token per row, and the rest of its sums into proj (window.hip)
int check_select_conv(const ChattsSelectArgs* a, const char* who);      // what chatts_select_conv takes (select.hip)
bool window_select_can_prep(const ChattsWindowArgs* w, const ChattsSelectArgs* c);
int window_select_prep(const ChattsWindowArgs* w, const ChattsSelectArgs* c, const SplitSums& in, float* proj, hipStream_t s);

constexpr int kRingPanel = 256;      // W rows per panel of the prefill kernel
// gemm_ring.hip: the prefill kernel's decomposition (M-tiles per panel, K splits) and launcher
struct RingGeom {
  int T, sk;          // M-tiles per panel, K splits
  int F, P;           // 16-row fragments of M, W panels
  int units;          // T * P * sk, ordered (split, panel, M-tile): the M-tiles of a panel are adjacent
  int wpx;            // workgroups per XCD (grid = 8 * wpx)
  int nf;             // a panel is 64 nf rows (3 or 4)
  int fbase, frem;    // fragments of an M-tile, the first frem tiles one more
  unsigned inv_t, inv_p;      // ceil(2^32 / T), / P, 0 for 1: a unit's place without divisions (units * T and * P are below 2^32)
  void finish() {
    fbase = F / T; frem = F % T;
    inv_t = T > 1 ? (unsigned)((0x100000000ull + T - 1) / T) : 0u;
    inv_p = P > 1 ? (unsigned)((0x100000000ull + P - 1) / P) : 0u;
  }
};
void ring_pick(int m, int n, int k, int cus, int force_t, int force_sk, int force_nf, RingGeom& g);
// the same kernel over lists of rows with weights of their own (experts): tiles [count][4] = {matrix, first place, places, -}, places of a tile
// at most kRingTile; order != nullptr: place -> row of A = order[place] / top, else A is packed by place.  C is packed by place; p.m: rows of A - 1 at most
struct RingGroup {
  const int32_t* tiles;
  const int32_t* count;      // device: number of tiles
  const int32_t* order;
  int top;
  int64_t w_stride;          // elements between matrices (p.w and p.wt)
};
constexpr int kRingTile = 160;
int launch_ring_group(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGroup& g, int most_tiles, hipStream_t s);
int launch_ring(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGeom& g, bool single, hipStream_t s);

// 1 / rms of the rows of A from the sums of squares that its producer left (GemmParams.row_ss: row r's parts at r * kSsStride): wave w takes rows
// w, w + waves, .. (ROWS of them).  Requested before anything else of the kernel and used at its end: a wait at the start would drain the first weights.
constexpr int kSsStride = 256;
template <int ROWS>
__device__ __forceinline__ void row_rstd_load(const GemmParams& p, int wave, int waves, int lane, f32x4 (&part)[ROWS]) {
  if (!p.row_ss) return;
#pragma unroll
  for (int t = 0; t < ROWS; ++t) part[t] = *reinterpret_cast<const f32x4*>(p.row_ss + ((wave + t * waves) & 15) * kSsStride + lane * 4);
}
template <int ROWS>
__device__ __forceinline__ void row_rstd_store(const GemmParams& p, int wave, int waves, int lane, const f32x4 (&part)[ROWS], float* rstd) {
  if (!p.row_ss) return;
#pragma unroll
  for (int t = 0; t < ROWS; ++t) {
    const int row = wave + t * waves;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) s += lane * 4 + j < p.row_ss_parts ? part[t][j] : 0.f;
    s = wave_sum(s);
    if (lane == 0 && row < 16) rstd[row] = rsqrtf(s / (float)p.k + p.row_eps);
  }
}

// gemm_rows.hip: few rows, whole K per workgroup
bool use_rows(const ChattsLinearArgs* a, int sk, bool hands_on);      // sk: K ranges of gemm_stream_kernel; hands_on: post_ss is asked for
int rows_grid(int n, int epilogue);      // workgroups = parts of post_ss
int launch_rows(const GemmParams& p, const ChattsLinearArgs* a, int sk, hipStream_t s);
// gemm_cols.hip: wide projections of few rows, K whole
bool use_cols(const ChattsLinearArgs* a);
int launch_cols(const GemmParams& p, const ChattsLinearArgs* a, hipStream_t s);
// chatts_rmsnorm_planes on rows that lie ldx apart (elementwise.hip)
int launch_rmsnorm_planes(const float* x, int ldx, const float* w, uint16_t* hi, uint16_t* lo, int ld_planes, int t, int hidden, float eps, int tiled, hipStream_t s);

// moe.hip: a feed-forward of the experts' kind beside them, for all rows, in their launches (2 to 16 rows): up as gate_up of an expert, f = its activations [rows, ff], y [rows, width_p]
struct MoeBeside {
  const chatts_bf16 *up, *up_t, *down, *down_t;
  int ff;
  chatts_bf16 *f_hi, *f_lo;
  float* y;
  float limit, alpha;      // CHATTS_EXPERT_CLAMPGLU
};
bool moe_takes_beside(const ChattsMoeArgs* a, const MoeBeside& sh);
// direct: no lists.  A pair of a row and a choice is its own place (row * top + choice; order, offsets and tiles are not read), an expert's launch blocks find its pairs in ids.  For 2 to 16 rows, up
// to 64 pairs and outputs, no choice groups (moe_takes_choice); ids, weight, place and kept then come from the norm before the router (depth.hip)
bool moe_takes_choice(const ChattsMoeArgs* a);
int depth_norm(const ChattsDepthNormArgs* a, bool tiles, chatts_stream_t stream);      // chatts_depth_norm; tiles: the operand's planes as plane_at has them, whole blocks of 16 rows in tiles
bool depth_norm_can_choose(int ldx, int router_rows, int outputs);
int depth_norm_choose(const ChattsDepthNormArgs* a, const ChattsMoeArgs* moe, const chatts_bf16* router, const chatts_bf16* router_t, int router_rows, chatts_stream_t stream);
int depth_norm_choose_sums(const ChattsDepthNormArgs* a, const ChattsMoeArgs* moe, const chatts_bf16* router, const chatts_bf16* router_t, int router_rows, const SplitSums* y,
                           chatts_stream_t stream);      // y: a->y as its projection's splits, or NULL
int moe_experts(const ChattsMoeArgs* a, const MoeBeside& sh, bool direct, chatts_stream_t stream);

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

}  // namespace chatts
