// gemv4_tiles.hip - projections of one row on 4-bit codes that were laid out once (chatts_tile_w4): out = epilogue(W . norm(x)).
//
// The weight is DEFINED as bf16_rne(code * scale - scale * zero).  gemv4_kernel (gemv4.hip) forms it on the vector pipe: v_fma_mix and v_cvt_pk issue at half rate, 3.6 issue slots a
// code, 13 of 20 us of a gate_up projection.  Here the matrix pipe multiplies by the scale, too:
//   * D = A . B + C with A = codes as float16 denormals (a mask makes two of them: code * 2^-24, or * 2^-20 for the nibble above), 16 places of K x 16 row slots, B = the slots' scales
//     on the diagonal (sixteen times them for the lower nibbles), C = -(scale * zero) * 2^-20: D holds weight * 2^-20 exactly (11 bits of a scale, 7 of code - zero), one v_cvt_pk rounds
//     two, and what is left are 1.6 slots a code.  The power of two is applied to the sums.
//   * a lane of A holds the codes of four rows at ONE place of K, which no row-major layout gives: the codes are stored in that order, units of four rows x 512 k = 1 KB that a wave
//     reads as one piece, and their 16 scales and zeros as 64 bytes.
//   * D is the operand of the second product as it lies: slots (4 rows x 4 parts of 128 k) x 8 places, against x as columns (part, hi / lo), as in gemv4_kernel.
// us there / here, both in one run, copies of the weights in turn (600 MB and more, so that they come from memory), the norm where the model has it, at 12 waves and a ring of four:
//   27648 x 5120 gated 22.5 / 17.5   24576 x 4096 gated 17.5 / 12.9   13824 x 5120 gated 12.7 / 10.2   16384 x 2048 gated 7.6 / 6.8   65536 x 8192 gated 78.3 / 53.2
//   5120 x 13824 13.4 / 10.9   4096 x 12288 11.3 / 8.6   5120 x 6912 7.5 / 7.3   2560 x 8192 7.2 / 6.9   2048 x 8192 5.7 / 5.8
//   7168 x 5120 8.7 / 7.3   6144 x 4096 6.7 / 6.2   3584 x 5120 6.5 / 5.9   5120 x 5120 6.9 / 6.4   4096 x 4096 5.5 / 5.1   5120 x 2560 5.2 / 4.8
// Another run of the same had up to 12 % more (27648 x 5120 18.4, 24576 x 4096 14.5): figures of one line belong together, those of different lines do not.  75 MB of 27648 x 5120 are 11.7 us
// at the rate of a stream; weights that lie in L2 or the Infinity Cache already are 0.2 to 0.9 faster: what is left is the launch, x and the conversion.
#include "common.h"
#include "gemv4.h"

namespace chatts {

typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int w4t_units(int k) { return (k + 511) >> 9; }      // of a quad of rows

struct W4TileParams {
  const uint8_t* w4;
  const float2* sz;
  int rows, k, ldw4, gshift, ng, gated;
  u32x4* codes;                       // [rows / 4][units][part][16] pieces
  uint32_t* scales;                   // [rows / 4][units][16]: float16 scale | float16 zero << 16
  int* bad;
};

// one wave per unit; lane: place i of 16, part of K
__global__ __launch_bounds__(256) void tile_w4_kernel(W4TileParams p) {
  const int S = w4t_units(p.k), unit = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63, i = lane & 15, part = lane >> 4;
  if (unit >= p.rows / 4 * S) return;
  const int quad = unit / S, s = unit - quad * S;
  auto row = [&](int r) {
    if (!p.gated) return quad * 4 + r;
    const int at = quad * 2;
    return (at >> 4) * 32 + (at & 15) + (r >> 1) + (r & 1) * 16;
  };
  auto code = [&](int r, int m) -> uint32_t {
    const int k = s * 512 + part * 128 + m * 16 + i;
    if (k >= p.k) return 0u;
    return (p.w4[(size_t)row(r) * p.ldw4 + (k >> 1)] >> ((k & 1) * 4)) & 15u;
  };
  u32x4 v;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    uint32_t w = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) w |= (code(r, 2 * d) | code(r, 2 * d + 1) << 4) << ((r & 1) * 16 + (r >> 1) * 8);
    v[d] = w;
  }
  p.codes[(size_t)unit * 64 + lane] = v;
  if (lane < 16) {
    const int k = s * 512 + (lane >> 2) * 128;
    uint32_t e = 0;
    if (k < p.k) {
      const float2 z = p.sz[(size_t)row(lane & 3) * p.ng + (k >> p.gshift)];
      const _Float16 h = (_Float16)z.x;
      const float zero = z.x == 0.f ? 0.f : rintf(z.y / z.x);
      const _Float16 zh = (_Float16)(-zero * 0x1p-20f);
      // (4000: sixteen times a scale has to be a float16 number)
      if (!(__builtin_isfinite(z.x) && (float)h == z.x && fabsf(zero) <= 64.f && (float)zh * z.x == -z.y * 0x1p-20f && fabsf(z.x) <= 4000.f)) atomicAdd(p.bad, 1);
      e = (uint32_t)__builtin_bit_cast(uint16_t, h) | (uint32_t)__builtin_bit_cast(uint16_t, zh) << 16;
    }
    p.scales[(size_t)unit * 16 + lane] = e;
  }
}

// us by waves / units of the ring, 8 / 3, 8 / 4, 12 / 3, 12 / 4, 16 / 3, one run:
//   65536 x 8192 gated 60.2, 58.4, 52.8, 52.5, no room   27648 x 5120 gated 19.3, 18.6, 17.8, 18.4, 17.5   13824 x 5120 gated 11.1, 11.2, 10.7, 10.5, 12.5   7168 x 5120 7.9, 7.8, 7.5, 7.5, 7.9
//   24576 x 4096 gated 14.0, 13.7, 14.3, 14.5, 14.2   5120 x 13824 11.6, 11.4, 11.7, 12.2, 12.3   4096 x 12288 9.2, 9.2, 9.1, 9.5, 9.9   5120 x 5120 6.2, 6.3, 6.0, 6.4, 6.8
//   16384 x 2048 gated 6.4, 6.8, 6.8, 7.0, 7.2   6144 x 4096 5.7, 5.8, 6.1, 6.2, 6.6   4096 x 4096 4.7, 4.8, 5.0, 5.1, 5.7   2560 x 8192 6.4, 6.4, 6.7, 6.9, 7.1   2048 x 8192 5.2, 5.2, 5.8, 5.9, 6.2
// Twelve are for K of 5120 and gated rows, where most of a ChatTS-14B step is; below 40 million codes eight are 3 to 12 % faster, and there is no rule between them yet.  A ring of eight units
// with eight waves takes 1 to 2 us more (every line of the unrolled loop is fetched by each launch).  More than one unit before x is there costs 0.2 to 0.9.
constexpr int kT4Bufs = 4, kT4Ahead = kT4Bufs - 1, kT4Waves = 12, kT4Threads = 64 * kT4Waves, kT4Turns = (16384 / 8 + kT4Threads - 1) / kT4Threads;

// weights of a unit, times 2^-20: the operands of four products of 32 k.  place 8 quad .. of product p: k = 16 ma + 4 quad .. + 3 and 32 further on, of this
// lane's part, ma = (p & 1) * 4 + (p >> 1)
struct W4Diag { uint32_t m0, m1; };
__device__ __forceinline__ W4Diag w4_diag(int lane) {
  const int j = lane & 15, q = lane >> 4, e = j & 3;
  const bool mine = q == j >> 2;
  return {mine && e < 2 ? 0xffffu << (e * 16) : 0u, mine && e >= 2 ? 0xffffu << ((e & 1) * 16) : 0u};
}
__device__ __forceinline__ void w4_weights(const u32x4 cv, const uint32_t sz, const W4Diag dg, bf16x8_t (&w)[4]) {
#ifdef __HIP_DEVICE_COMPILE__
  const f16x2_t h = __builtin_bit_cast(f16x2_t, sz), sx = {h.x, h.x}, s16 = sx * (_Float16)16.f;
  const uint32_t s2 = __builtin_bit_cast(uint32_t, sx), t2 = __builtin_bit_cast(uint32_t, s16);
  const f16x4_t b = __builtin_bit_cast(f16x4_t, (u32x2){s2 & dg.m0, s2 & dg.m1}), b16 = __builtin_bit_cast(f16x4_t, (u32x2){t2 & dg.m0, t2 & dg.m1});
  const float nz = (float)h.x * (float)h.y;
  const f32x4 c0 = {nz, nz, nz, nz};
  f32x4 de[4], d1[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t v = cv[d], u = v >> 8;
    de[d] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, (u32x2){v & 0x000f000fu, u & 0x000f000fu}), b16, c0, 0, 0, 0);
    d1[d] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, (u32x2){v & 0x00f000f0u, u & 0x00f000f0u}), b, c0, 0, 0, 0);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w[p][e] = (__bf16)de[2 * p][e];
      w[p][4 + e] = (__bf16)de[2 * p + 1][e];
      w[2 + p][e] = (__bf16)d1[2 * p][e];
      w[2 + p][4 + e] = (__bf16)d1[2 * p + 1][e];
    }
#endif
}

template <int EPI, bool NORM>
__global__ __launch_bounds__(64 * kT4Waves) void gemv4_tiles_kernel(Gemv4Params p) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float red[kT4Waves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = p.k, S = w4t_units(K), b0 = (int)blockIdx.x;
  const int q0 = b0 * p.quads_each + (b0 < p.quads_more ? b0 : p.quads_more), nq = p.quads_each + (b0 < p.quads_more);
  char* xs = smem;                                                       // [S * 4] operands
  f32x4* part = reinterpret_cast<f32x4*>(smem + (size_t)S * 4 * kQ4Piece);      // [quad][wave][8]
  const int items = nq * S, i0 = wave * items / kT4Waves, cnt = (wave + 1) * items / kT4Waves - i0;
  const int kq = lane >> 4, col = lane & 15;
  const W4Diag dg = w4_diag(lane);
  const unsigned units = (unsigned)(p.n >> 2) * (unsigned)S;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.w4, 0, (int)(units * 1024u), 0x00020000);
  const __amdgpu_buffer_rsrc_t zr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w4 + (size_t)units * 1024u), 0, (int)(units * 64u), 0x00020000);
  u32x4 cv[kT4Bufs];
  uint32_t zv[kT4Bufs];
  unsigned at = (unsigned)(q0 * S + i0);                                 // the unit to request next
  const unsigned end = at + (unsigned)cnt;
  auto request = [&](int b) __attribute__((always_inline)) {             // (past the share: outside the buffer, nothing returns)
    const unsigned u = at < end ? at : 0x1fffffu;
    cv[b] = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)(lane * 16u + u * 1024u), 0, 2 /* nt: streamed once */);
    zv[b] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(zr, (int)(col * 4u + u * 64u), 0, 2);
    ++at;
  };
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, K * 4, 0x00020000);      // (past K: zeros)
  const __amdgpu_buffer_rsrc_t nr = __builtin_amdgcn_make_buffer_rsrc((void*)(NORM ? p.norm_w : p.x), 0, K * 4, 0x00020000);
  f32x4 xv[kT4Turns][2], gw[kT4Turns][2];
  // item of x: unit, part, product, quad of lanes: k of its first four, the others 32 further on
  auto item_k = [&](int it) { return (it >> 6) * 512 + ((it >> 4) & 3) * 128 + ((it >> 3) & 1) * 64 + ((it >> 2) & 1) * 16 + (it & 3) * 4; };
#pragma unroll
  for (int j = 0; j < kT4Turns; ++j)
    if (j * kT4Threads * 8 < K) {
      const int k = item_k(tid + j * kT4Threads);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        xv[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, k * 4 + 128 * i, 0, 0));
        if (NORM) gw[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(nr, k * 4 + 128 * i, 0, 0));
      }
    }
  __builtin_amdgcn_sched_barrier(0);
  request(0);
  __builtin_amdgcn_sched_barrier(0);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kT4Turns; ++j)
    if (j * kT4Threads * 8 < K) {
#pragma clang fp contract(off)      // lo is the split of the ROUNDED product
      const int it = tid + j * kT4Threads;
      bf16x8_t hi, lo;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (NORM) ss = sumsq4(ss, xv[j][i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = xv[j][e >> 2][e & 3];
        if (NORM) v *= gw[j][e >> 2][e & 3];
        const __bf16 h = (__bf16)v;
        hi[e] = h;
        lo[e] = (__bf16)(v - (float)h);
      }
      if (it < S * 64) {
        const int pr = ((it >> 3) & 1) + ((it >> 2) & 1) * 2;            // product: ma = (pr & 1) * 4 + (pr >> 1)
        char* to = xs + ((it >> 6) * 4 + pr) * kQ4Piece + ((it & 3) * 8 + ((it >> 4) & 3) * 2) * 16;
        *reinterpret_cast<bf16x8_t*>(to) = hi;
        *reinterpret_cast<bf16x8_t*>(to + 16) = lo;
      }
    }
  if (NORM) {                              // the factor 1 / rms is applied to the sums: x need not wait for it
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
  }
#pragma unroll
  for (int b = 1; b < kT4Ahead; ++b) request(b);
  __syncthreads();

  int q = i0 / S, s = i0 - q * S;                                        // the unit to compute next
  f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
  auto flush = [&]() __attribute__((always_inline)) {                    // rows 4 kq .. of the product belong to part kq: columns 2 kq and 2 kq + 1 are theirs
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (acc0[j] + acc1[j]) * 0x1p20f;
    if ((col >> 1) == kq) part[(q * kT4Waves + wave) * 8 + col] = v;
    acc0 = acc1 = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  const char* xl = xs + (kq * 8 + (lane & 7)) * 16;
  // A SIMD issues for its oldest wave first: of three waves with equal shares of 27648 x 5120 the first was done at 12.5 us, the last at 21.  A wave that is ahead lets the others go first:
  // 15.1 and 18.6.  us without / with, one run: 27648 x 5120 gated 19.8 / 18.4, 65536 x 8192 gated 55.6 / 52.5, 13824 x 5120 gated 11.4 / 10.5, 5120 x 13824 12.6 / 12.2, 7168 x 5120 7.7 / 7.5,
  // nothing for shares of few units (0.1 to either side).
  int calm = 0, level = 3;
  for (int t = 0; t < cnt; t += kT4Bufs) {
    if (t >= calm) {
      if (level == 3) __builtin_amdgcn_s_setprio(3);
      else if (level == 2) __builtin_amdgcn_s_setprio(2);
      else if (level == 1) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
      --level;
      calm += (cnt + 3) >> 2;
    }
#pragma unroll
    for (int b = 0; b < kT4Bufs; ++b) {
      request((b + kT4Ahead) % kT4Bufs);
      __builtin_amdgcn_sched_barrier(0);
      if (t + b < cnt) {
        bf16x8_t w[4];
        w4_weights(cv[b], zv[b], dg, w);
        const char* xp = xl + s * 4 * kQ4Piece;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[m], *reinterpret_cast<const bf16x8_t*>(xp + m * kQ4Piece), acc0, 0, 0, 0);
          acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 + m], *reinterpret_cast<const bf16x8_t*>(xp + (2 + m) * kQ4Piece), acc1, 0, 0, 0);
        }
        if (++s == S) { flush(); s = 0; ++q; }
      }
    }
  }
  if (cnt > 0 && s > 0) flush();
  __syncthreads();
  q4_finish<EPI, NORM, kT4Waves>(p, part, red, tid, q0, nq, S, items);
#endif
}

template <int EPI, bool NORM>
static int launch4t_t(const Gemv4Params& p, int grid, size_t lds, hipStream_t s) {
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv4_tiles_kernel<EPI, NORM>), hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemv4_tiles: cannot reserve 156 KB of LDS: %s", hipGetErrorString(e));
    configured = true;
  }
  hipLaunchKernelGGL((gemv4_tiles_kernel<EPI, NORM>), dim3(grid), dim3(64 * kT4Waves), lds, s, p);
  CHATTS_CHECK_LAUNCH("gemv4_tiles");
  return CHATTS_OK;
}
template <int EPI>
static int launch4t_e(const Gemv4Params& p, int grid, size_t lds, hipStream_t s) {
  return p.norm_w ? launch4t_t<EPI, true>(p, grid, lds, s) : launch4t_t<EPI, false>(p, grid, lds, s);
}

int launch_gemv4_tiles(const ChattsLinearArgs* a, const void* tiles, hipStream_t s) {
  Gemv4Params p{};
  p.w4 = static_cast<const uint8_t*>(tiles); p.x = a->a; p.norm_w = a->norm_w; p.bias = a->bias; p.resid = a->resid; p.out = a->c; p.eps = a->norm_eps;
  p.n = a->n; p.k = a->k;
  const int quads = a->n / 4, cus = device_cus(), grid = quads < cus ? quads : cus;
  p.quads_each = quads / grid; p.quads_more = quads % grid;
  const size_t lds = q4_lds(a->k, (quads + grid - 1) / grid, kT4Waves);
  switch (a->epilogue) {
    case CHATTS_EPI_RESID: return launch4t_e<CHATTS_EPI_RESID>(p, grid, lds, s);
    case CHATTS_EPI_SWIGLU: return launch4t_e<CHATTS_EPI_SWIGLU>(p, grid, lds, s);
    default: return launch4t_e<CHATTS_EPI_NONE>(p, grid, lds, s);
  }
}

}  // namespace chatts

using namespace chatts;

// Short rows of few codes keep the row-major kernels: 4.2 us here before any code is read, 3 there.  us there / here: 1024 x 512 3.0 / 4.3, 4096 x 1024 3.8 / 4.3, 8192 x 1024 4.5 / 4.8, 2048 x 2048
// 3.9 / 4.2, 1536 x 2560 5.1 / 5.1, 1024 x 4096 4.7 / 4.7; but 16384 x 1024 gated 5.6 / 5.6, 3072 x 3072 5.2 / 4.7, 4096 x 2560 5.2 / 4.5, 6144 x 2048 5.6 / 5.2.  Left over: 2048 x 8192 (3 %).
extern "C" size_t chatts_tile_w4_bytes(int rows, int k, int group) {
  if (rows < 16 || rows % 16 || k < 128 || k > 16384 || group < 128 || (group & (group - 1)) || k % group || (size_t)rows * k <= (size_t)1 << 23) return 0;
  const size_t units = (size_t)rows / 4 * w4t_units(k);
  const int quads = rows / 4, cus = device_cus();
  if (units * 1024 >= (size_t)kQ4Far - 4096 || cus < 1 || q4_lds(k, (quads + cus - 1) / cus, kT4Waves) > 156 * 1024) return 0;
  return units * (1024 + 64);
}

extern "C" int chatts_tile_w4(const uint8_t* w4, const float* w4_sz, int rows, int k, int ldw4, int group, int gated, void* dst, int32_t* bad, chatts_stream_t stream) {
  CHATTS_REQUIRE(w4 && w4_sz && dst && bad, CHATTS_E_BADARG, "tile_w4: null pointer");
  CHATTS_REQUIRE(chatts_tile_w4_bytes(rows, k, group) != 0 && ldw4 >= k / 2 && (!gated || rows % 32 == 0) && ((uintptr_t)dst % 16) == 0 && ((uintptr_t)w4_sz % 8) == 0 && ((uintptr_t)bad % 4) == 0,
                 CHATTS_E_SHAPE, "tile_w4: %d x %d in groups of %d has no tiled form", rows, k, group);
  W4TileParams p;
  p.w4 = w4; p.sz = reinterpret_cast<const float2*>(w4_sz); p.rows = rows; p.k = k; p.ldw4 = ldw4; p.gshift = 31 - __builtin_clz(group); p.ng = k / group; p.gated = gated;
  const size_t units = (size_t)rows / 4 * w4t_units(k);
  p.codes = static_cast<u32x4*>(dst); p.scales = reinterpret_cast<uint32_t*>(static_cast<char*>(dst) + units * 1024); p.bad = bad;
  hipLaunchKernelGGL(tile_w4_kernel, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, as_stream(stream), p);
  CHATTS_CHECK_LAUNCH("tile_w4");
  return CHATTS_OK;
}

extern "C" int chatts_linear_w4_tiles(const ChattsLinearArgs* a, const void* tiles, chatts_stream_t stream) {
  CHATTS_REQUIRE(a && tiles && a->a && a->c && a->m == 1 && a->batch <= 1 && !a->tp_reduce && !a->c_hi && !a->post_norm_w && !a->a_hi && !a->exact_f32, CHATTS_E_BADARG,
                 "linear_w4_tiles: one row of float32 A and C, without planes, exchange or batch");
  CHATTS_REQUIRE(a->n > 0 && a->k > 0 && chatts_tile_w4_bytes(a->n, a->k, 128) != 0, CHATTS_E_SHAPE, "linear_w4_tiles: %d x %d has no tiled form", a->n, a->k);
  CHATTS_REQUIRE(a->epilogue == CHATTS_EPI_NONE || (a->epilogue == CHATTS_EPI_RESID && a->resid) || (a->epilogue == CHATTS_EPI_SWIGLU && a->n % 32 == 0), CHATTS_E_BADARG,
                 "linear_w4_tiles: epilogue %d", a->epilogue);
  CHATTS_REQUIRE(((uintptr_t)a->a % 16) == 0 && ((uintptr_t)a->c % 16) == 0 && ((uintptr_t)tiles % 16) == 0, CHATTS_E_SHAPE, "linear_w4_tiles: pointers must be 16-byte aligned");
  return launch_gemv4_tiles(a, tiles, as_stream(stream));
}
