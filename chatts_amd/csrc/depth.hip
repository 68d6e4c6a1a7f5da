// depth.hip - the residual stream of layers with norms before their sublayers only: a sublayer's share (its output, the experts' weighted sum) enters x
// with a factor, the streams of all earlier layers are averaged, and the next norm's operand leaves in the same launch, a workgroup per row.
// Also the cap of the logits.
#include "gemm_common.h"
#include "moe_route.h"

namespace chatts {

// The router behind the norm: logits of NR x 16 outputs and the row's choice.  w: [16 NR][ldx], row-major (step 1) or chatts_tile_bf16's copy of it (step 16: a K-step is 1 KB further)
struct DepthChoose {
  const uint16_t* w;
  int step;
  ChattsMoeArgs moe;
};

// a thread keeps its columns in registers.  NT: threads (more of them for a few rows: then every load of a row is in flight at once)
// NR > 0 (2 to 16 rows): the same launch multiplies the row by the router, as the planes that it writes, and chooses its experts.  A projection, its split's epilogue and a workgroup that chose
// for all rows and made lists of them were three launches: 12.5 us a layer of 32 experts at 16 rows of 2048, now 1.  The router's first K-steps are requested before the row is there.
// S_IN: y is what its projection left, up to so many splits, all requested with the row (16 rows of 2048, eight splits or sixteen: a layer's launch less, 921 -> 911 us a step of eight layers)
template <int NT, int NV, int NR = 0, int S_IN = 0>
__global__ __launch_bounds__(NT) void depth_norm_kernel(ChattsDepthNormArgs p, DepthChoose ch, int tiled, SplitSums y_in) {
  kernarg_touch<sizeof(ChattsDepthNormArgs) + sizeof(DepthChoose) + (S_IN ? 8 + sizeof(SplitSums) : 4)>();
  __shared__ float red[NT / 64];
  constexpr int NW = NT / 64, NX = NV * NT * 4;
  __shared__ __attribute__((aligned(16))) uint16_t xh[NR ? NX : 1], xl[NR ? NX : 1];
  __shared__ __attribute__((aligned(16))) float part[NR ? NW : 1][NR ? NR * 16 : 1];
  const size_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, fg = lane >> 4, steps = p.ldx >> 5;
  const uint16_t* rw = NR ? ch.w + (ch.step == 1 ? (size_t)fr * p.ldx + fg * 8 : (size_t)(fr * 4 + (fg ^ ((fr >> 3) << 1))) * 8) : nullptr;
  constexpr int RU = 4;      // K-steps of a wave requested at once: wave, wave + NW, ..
  bf16x8_t wf[NR ? RU : 1][NR ? NR : 1];
  auto request = [&](int s0) {
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int s = s0 + u * NW < steps ? s0 + u * NW : wave < steps ? wave : 0;
#pragma unroll
      for (int f = 0; f < NR; ++f) wf[u][f] = *reinterpret_cast<const bf16x8_t*>(rw + (size_t)f * 16 * p.ldx + (size_t)s * 32 * ch.step);
    }
  };
  if constexpr (NR > 0) request(wave);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = NV <= 2 ? 4 : 2;      // rows requested at once
  f32x4 x[NV], add[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * NT + tid) * 4;
    x[i] = c < p.ldx ? *reinterpret_cast<const f32x4*>(p.x + row * p.ldx + c) : zero;
    if constexpr (S_IN > 0) add[i] = c < p.ldx ? split_sum4<S_IN>(y_in, (int)row, c) : zero;
    else add[i] = p.y && c < p.ldx ? *reinterpret_cast<const f32x4*>(p.y + row * p.ldx + c) : zero;
  }
  if (p.ey) {
    for (int j0 = 0; j0 < p.top; j0 += U) {
      int at[U];
      float f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u < p.top ? j0 + u : j0;
        at[u] = j0 + u < p.top ? p.place[row * p.top + j] : -1;      // (uniform)
        f[u] = p.weight[row * p.top + j];
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = (i * NT + tid) * 4;
        if (c >= p.ldx) continue;
        f32x4 y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] = at[u] >= 0 ? *reinterpret_cast<const f32x4*>(p.ey + (size_t)at[u] * p.ldx + c) : zero;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) add[i][k] += at[u] >= 0 ? f[u] * y[u][k] : 0.f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) x[i][k] += p.mult * add[i][k];
  if (p.depth) {
    const float own = p.depth[p.n_streams];
    float* st = p.streams + row * p.ldx;
    if (p.keep) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = (i * NT + tid) * 4;
        if (c < p.ldx) *reinterpret_cast<f32x4*>(st + p.n_streams * p.stream_stride + c) = x[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) x[i][k] *= own;
    for (int j0 = 0; j0 < p.n_streams; j0 += U) {
      float f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] = j0 + u < p.n_streams ? p.depth[j0 + u] : 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = (i * NT + tid) * 4;
        if (c >= p.ldx) continue;
        f32x4 s[U];
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = j0 + u < p.n_streams ? *reinterpret_cast<const f32x4*>(st + (j0 + u) * p.stream_stride + c) : zero;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < 4; ++k) x[i][k] += f[u] * s[u][k];
      }
    }
  }
  if (p.y || p.ey || p.depth) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * NT + tid) * 4;
      if (c < p.ldx) *reinterpret_cast<f32x4*>(p.x + row * p.ldx + c) = x[i];
    }
  }
  if (!p.w) return;
  f32x4 w[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * NT + tid) * 4;
    w[i] = c < p.ldx ? *reinterpret_cast<const f32x4*>(p.w + c) : zero;      // (the weights travel while the row is reduced)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c + k < p.width) ss += x[i][k] * x[i][k];
  }
  ss = block_sum<NT / 64>(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)p.width + p.eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * NT + tid) * 4;
    if (c >= p.ldx) continue;
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = c + k < p.width ? x[i][k] * inv * w[i][k] : 0.f;
    if (NR == 0 && tiled) {      // (rows from `tiled` on: plane_at has them where row-major has)
      ChattsOperand at{};
      const size_t place = plane_at((int)row, c, p.ldx, tiled);
      at.hi = p.out.hi + place; at.lo = p.out.lo + place;
      store_operand4(at, 0, 0, v);
    } else {
      store_operand4(p.out, row, c, v);
    }
    if constexpr (NR > 0) {
      ChattsOperand own{};
      own.hi = xh; own.lo = xl;
      store_operand4(own, 0, c, v);
    }
  }
  if constexpr (NR > 0) {
    __syncthreads();
    f32x4 acc[NR];
#pragma unroll
    for (int f = 0; f < NR; ++f) acc[f] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave; s0 < steps; s0 += RU * NW) {
      if (s0 != wave) request(s0);
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const int s = s0 + u * NW;
        if (s >= steps) break;      // (uniform)
        const bf16x8_t h = *reinterpret_cast<const bf16x8_t*>(xh + s * 32 + fg * 8), l = *reinterpret_cast<const bf16x8_t*>(xl + s * 32 + fg * 8);      // (the row in every column)
#pragma unroll
        for (int f = 0; f < NR; ++f) {
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][f], l, acc[f], 0, 0, 0);
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][f], h, acc[f], 0, 0, 0);
        }
      }
    }
    if (fr == 0)
#pragma unroll
      for (int f = 0; f < NR; ++f) *reinterpret_cast<f32x4*>(&part[wave][f * 16 + fg * 4]) = acc[f];
    __syncthreads();
    if (wave) return;
    float z = 0.f;
    if (lane < NR * 16)
#pragma unroll
      for (int i = 0; i < NW; ++i) z += part[i][lane];
    const int id = moe_route_row64(ch.moe, (int)row, lane, z);
    if (lane < ch.moe.top) ch.moe.place[row * ch.moe.top + lane] = id >= 0 ? (int)row * ch.moe.top + lane : -1;
  }
}

__global__ __launch_bounds__(256) void soft_cap_kernel(float* __restrict__ x, int64_t quads, int64_t n, float cap, float k) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  auto f = [&](float v) { return cap - 2.f * cap * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(v * k)); };
  if (i < quads) {
    f32x4 v = *reinterpret_cast<const f32x4*>(x + i * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = f(v[j]);
    *reinterpret_cast<f32x4*>(x + i * 4) = v;
  } else if (i == quads) {
    for (int64_t j = quads * 4; j < n; ++j) x[j] = f(x[j]);
  }
}

}  // namespace chatts

using namespace chatts;

static int check_depth_norm(const ChattsDepthNormArgs* a) {
  CHATTS_REQUIRE(a && a->x && a->t >= 0 && a->width > 0, CHATTS_E_BADARG, "depth_norm: bad arguments");
  CHATTS_REQUIRE(a->ldx >= a->width && a->ldx % 4 == 0 && a->ldx <= 16384, CHATTS_E_SHAPE, "depth_norm: a width of %d in rows of %d (at most 16384)", a->width, a->ldx);
  CHATTS_REQUIRE(!a->ey || (a->place && a->weight && a->top > 0), CHATTS_E_BADARG, "depth_norm: experts");
  CHATTS_REQUIRE(!a->depth || (a->n_streams >= 0 && (a->streams || (a->n_streams == 0 && !a->keep)) && a->stream_stride % 4 == 0), CHATTS_E_BADARG,
                 "depth_norm: an average over %d streams", a->n_streams);
  CHATTS_REQUIRE(!a->w || ((a->out.f32 || a->out.hi) && a->out.ld >= a->ldx && a->out.ld % 4 == 0), CHATTS_E_SHAPE, "depth_norm: operand rows of %d", a->out.ld);
  CHATTS_REQUIRE((((uintptr_t)a->x | (uintptr_t)a->y | (uintptr_t)a->ey | (uintptr_t)a->w | (uintptr_t)a->streams | (uintptr_t)a->out.f32) % 16) == 0 &&
                     (((uintptr_t)a->out.hi | (uintptr_t)a->out.lo) % 8) == 0, CHATTS_E_SHAPE, "depth_norm: pointers must be aligned (16 bytes, planes 8)");
  return CHATTS_OK;
}
extern "C" int chatts_depth_norm(const ChattsDepthNormArgs* a, chatts_stream_t stream) { return depth_norm(a, false, stream); }
int chatts::depth_norm(const ChattsDepthNormArgs* a, bool tiles, chatts_stream_t stream) {
  if (const int rc = check_depth_norm(a)) return rc;
  CHATTS_REQUIRE(!tiles || (a->w && a->out.hi && a->out.lo && !a->out.f32 && a->out.ld == a->ldx && a->ldx % 32 == 0), CHATTS_E_SHAPE, "depth_norm: planes in tiles of %d columns", a->ldx);
  if (a->t == 0) return CHATTS_OK;
  const int tiled = tiles ? a->t & ~15 : 0;
  const DepthChoose none{};
  const dim3 g(a->t);
  hipStream_t s = as_stream(stream);
  if (a->ldx <= 1024) hipLaunchKernelGGL((depth_norm_kernel<256, 1>), g, dim3(256), 0, s, *a, none, tiled, SplitSums{});
  else if (a->t <= 64 && a->ldx <= 4096) hipLaunchKernelGGL((depth_norm_kernel<1024, 1>), g, dim3(1024), 0, s, *a, none, tiled, SplitSums{});
  else if (a->t <= 64 && a->ldx <= 8192) hipLaunchKernelGGL((depth_norm_kernel<1024, 2>), g, dim3(1024), 0, s, *a, none, tiled, SplitSums{});
  else if (a->ldx <= 2048) hipLaunchKernelGGL((depth_norm_kernel<256, 2>), g, dim3(256), 0, s, *a, none, tiled, SplitSums{});
  else if (a->ldx <= 4096) hipLaunchKernelGGL((depth_norm_kernel<256, 4>), g, dim3(256), 0, s, *a, none, tiled, SplitSums{});
  else if (a->ldx <= 8192) hipLaunchKernelGGL((depth_norm_kernel<256, 8>), g, dim3(256), 0, s, *a, none, tiled, SplitSums{});
  else hipLaunchKernelGGL((depth_norm_kernel<1024, 4>), g, dim3(1024), 0, s, *a, none, tiled, SplitSums{});
  CHATTS_CHECK_LAUNCH("depth_norm");
  return CHATTS_OK;
}

// ... and the choice of experts for rows that moe_takes_choice: ids, weight, place (a pair's own) and kept
// (a router of router_rows x ldx, outputs of them in use: the kernel reads 32 rows or 64)
static int router_blocks(int outputs) { return outputs <= 32 ? 2 : 4; }
bool chatts::depth_norm_can_choose(int ldx, int router_rows, int outputs) { return ldx % 64 == 0 && ldx <= 4096 && outputs <= 64 && router_rows >= 16 * router_blocks(outputs); }
// (rows that are there already; the tests call it)
int chatts::depth_norm_choose(const ChattsDepthNormArgs* a, const ChattsMoeArgs* moe, const chatts_bf16* router, const chatts_bf16* router_t, int router_rows, chatts_stream_t stream) {
  return depth_norm_choose_sums(a, moe, router, router_t, router_rows, nullptr, stream);
}
int chatts::depth_norm_choose_sums(const ChattsDepthNormArgs* a, const ChattsMoeArgs* moe, const chatts_bf16* router, const chatts_bf16* router_t, int router_rows, const SplitSums* y,
                                   chatts_stream_t stream) {
  if (const int rc = check_depth_norm(a)) return rc;
  CHATTS_REQUIRE(moe && router && a->w && a->out.hi && a->out.lo && depth_norm_can_choose(a->ldx, router_rows, moe->experts + moe->identity) && moe_takes_choice(moe) &&
                     moe->n_rows == a->t && moe->ids && moe->place && moe->weight && moe->kept && moe->rows && ((uintptr_t)router % 16) == 0 && ((uintptr_t)router_t % 16) == 0, CHATTS_E_BADARG, "depth_norm: a choice behind %d rows of %d", a->t, a->ldx);
  if (a->t == 0) return CHATTS_OK;
  const DepthChoose ch{router_t ? router_t : router, router_t ? 16 : 1, *moe};
  CHATTS_REQUIRE(!y || (a->y && y->sk >= 1 && y->sk <= kMostNormSums && y->n == a->ldx), CHATTS_E_SHAPE, "depth_norm: %d splits of %d columns", y->sk, y->n);
  const SplitSums in = y ? *y : SplitSums{};
#define CHATTS_CHOOSE(R, S) hipLaunchKernelGGL((depth_norm_kernel<1024, 1, R, S>), dim3(a->t), dim3(1024), 0, as_stream(stream), *a, ch, 0, in)
  if (router_blocks(moe->experts + moe->identity) == 2) {
    if (!y) CHATTS_CHOOSE(2, 0); else if (in.sk <= 8) CHATTS_CHOOSE(2, 8); else CHATTS_CHOOSE(2, kMostNormSums);
  } else {
    if (!y) CHATTS_CHOOSE(4, 0); else if (in.sk <= 8) CHATTS_CHOOSE(4, 8); else CHATTS_CHOOSE(4, kMostNormSums);
  }
#undef CHATTS_CHOOSE
  CHATTS_CHECK_LAUNCH("depth_norm_choose");
  return CHATTS_OK;
}

extern "C" int chatts_soft_cap(float* x, int64_t n, float cap, chatts_stream_t stream) {
  CHATTS_REQUIRE(x && n >= 0 && cap > 0.f && ((uintptr_t)x % 16) == 0, CHATTS_E_BADARG, "soft_cap: %lld values, cap %g", (long long)n, (double)cap);
  if (n == 0) return CHATTS_OK;
  const int64_t quads = n / 4;
  hipLaunchKernelGGL(soft_cap_kernel, dim3((unsigned)((quads + 1 + 255) / 256)), dim3(256), 0, as_stream(stream), x, quads, n, cap, 2.0f * 1.44269504088896341f / cap);
  CHATTS_CHECK_LAUNCH("soft_cap");
  return CHATTS_OK;
}
