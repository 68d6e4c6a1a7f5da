// gemv4.hip - the batch-1 projection on 4-bit codes (GPTQ format) with the matrix pipe: out = epilogue(W . norm(x)), W rebuilt from codes.
//
// The weight is DEFINED as bf16_rne(code * scale - scale * zero), so every code costs its own conversion: the kernel is bound by vector operations and
// by HBM at about the same time, and gains from doing less per code and from doing both at once.  gemv4_ldsx_kernel (gemv.hip) spends 3.75
// operations a code and waits for a batch of loads before it computes on it.  Here:
//   * conversion: nibbles 0 and 4 (1 and 5, ...) of a word masked in place ARE two float16 denormals, code * 2^-24 (or * 2^-20), so one v_fma_mix each
//     with scale * 2^24 gives code * scale - scale * zero with a single rounding (scales below 2^104; sums that are not finite are done again code by code), and v_cvt_pk rounds two of them:
//     2.1 operations a code; the order of k that falls out (0 4 1 5 2 6 3 7) is x's order in LDS;
//   * products on the matrix pipe: a wave's unit is FOUR rows ("quad") x 512 k, one 16-byte load per lane = 256 consecutive bytes of each row.  The 16
//     rows of an MFMA operand are 4 rows x 4 parts of K; x comes as columns (part, hi / lo), and the wanted sums are the blocks where the parts
//     agree: nothing is wasted on rows that are not there, and a wave ends up with 8 vectors of 4 rows instead of a 64-lane reduction;
//   * the quads of a workgroup (one per CU, N / 4 / 256 of them) x the parts of K are dealt evenly over 8 waves, loads two units ahead and the first
//     ones before x is staged; requests past the end of a wave's share carry an offset outside the buffer: they return nothing.
// Measured back to back in a graph, there -> here: qkv 7168 x 5120 10.8 -> 8.4 us, o 5120 x 5120 8.7 -> 7.4, gate_up 27648 x 5120 27.9 -> 19.9 (75 MB with scales:
// 3.8 TB/s; v_fma_mix and v_cvt_pk issue at half rate, so the conversion alone is 13 us of it), down 5120 x 13824 17.0 -> 12.2.  16 waves instead of 8: 1 us
// more everywhere (the prologue is serial per SIMD); scales staged in LDS: 1 to 2 us more.
// x = hi + lo bf16 (2^-17), products exact, float32 sums: the accuracy of the kernel it replaces.
#include <type_traits>

#include "gemv4.h"

namespace chatts {

// Units of the ring: more of them only cost code and registers.  us with 8 / 6 / 4 / 3 / 2: 7168 x 5120 9.9 / 9.1 / 9.0 / 8.4 / 9.3, 5120 x 5120 8.5 / 8.2 / 7.4 / 7.4 / 7.7, 27648 x 5120 gated
// 21.5 / 20.3 / 20.2 / 19.9 / 22.4, 5120 x 13824 13.9 / 12.6 / 12.6 / 12.2 / 13.7, 24576 x 4096 gated 17.0 / 16.4 / 15.3 / 15.2 / 16.4, 4096 x 12288 11.5 / 10.3 / 9.9 / 10.0 / 10.8.
constexpr int kQ4Bufs = 3, kQ4Ahead = kQ4Bufs - 1;

template <int EPI, bool NORM>
__global__ __launch_bounds__(64 * kQ4Waves) void gemv4_kernel(Gemv4Params p) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float red[kQ4Waves];
  constexpr bool GLU = epi_is_glu(EPI);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = p.k, S = q4_parts(K), b0 = (int)blockIdx.x;
  const int q0 = b0 * p.quads_each + (b0 < p.quads_more ? b0 : p.quads_more), nq = p.quads_each + (b0 < p.quads_more);
  char* xs = smem;                                                       // [S * 4] operands
  f32x4* part = reinterpret_cast<f32x4*>(smem + (size_t)S * 4 * kQ4Piece);      // [quad][wave][8]
  const int items = nq * S, i0 = wave * items / kQ4Waves, cnt = (wave + 1) * items / kQ4Waves - i0;

  // lane: row r of the quad, part kap of K within the unit, k group kq of 32 codes within the part
  const int r = lane & 3, kap = (lane >> 2) & 3, kq = lane >> 4, pos = kap * 4 + kq;
  // (up to the last code of the last row: units of 512 codes run past the end of a row)
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.w4, 0, (int)((unsigned)(p.n - 1) * (unsigned)p.ldw4 + (unsigned)K / 2u), 0x00020000);
  const unsigned lane_off = (unsigned)(GLU ? (r >> 1) + (r & 1) * 16 : r) * (unsigned)p.ldw4 + pos * 16;
  auto first_row = [&](int q) __attribute__((always_inline)) { return q4_first_row<GLU>(q0 + q); };
  // scale and zero of this lane's 32 codes: they lie in one group, and 512 s is a whole number of groups or inside one
  const __amdgpu_buffer_rsrc_t zr = __builtin_amdgcn_make_buffer_rsrc((void*)p.sz, 0, (int)((unsigned)p.n * (unsigned)p.ng * 8u), 0x00020000);
  const unsigned lane_sz = ((unsigned)(GLU ? (r >> 1) + (r & 1) * 16 : r) * (unsigned)p.ng + (unsigned)((pos * 32) >> p.gshift)) * 8u;
  const unsigned lane_sz_end = (S - 1) * 512 + pos * 32 < K ? lane_sz : kQ4Far;      // past K: scale and zero read as 0, so weights of 0 (the codes are the next row's)
  u32x4 cv[kQ4Bufs];
  u32x2 zv[kQ4Bufs];
  const int first_q = p.parts_inv ? (int)__umulhi((unsigned)i0, p.parts_inv) : i0;
  int rq = first_q, rs = i0 - rq * S, ri = 0;                            // the unit to request next
  int q = rq, s = rs;                                                    // ... and the one to compute next
  auto request = [&](int b) __attribute__((always_inline)) {
    const unsigned row = (unsigned)first_row(rq);
    const unsigned at = ri < cnt ? row * (unsigned)p.ldw4 + (unsigned)rs * 256u : kQ4Far, zat = ri < cnt ? (row * (unsigned)p.ng + (unsigned)((rs * 512) >> p.gshift)) * 8u : kQ4Far;
    cv[b] = __builtin_amdgcn_raw_buffer_load_b128(wr, lane_off + at, 0, 2 /* nt: streamed once */);
    zv[b] = __builtin_amdgcn_raw_buffer_load_b64(zr, (rs == S - 1 ? lane_sz_end : lane_sz) + zat, 0, 0);
    ++ri;
    if (++rs == S) { rs = 0; ++rq; }
  };
  // x: eight k a thread and turn, times the norm's weights, split, written as operands.  It is requested before the weights (loads return in order: x comes from
  // L2, weights from HBM), and only one unit of those before it is there: more would stand in front of the x that later waves ask for.
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, K * 4, 0x00020000);      // (past K: zeros)
  const __amdgpu_buffer_rsrc_t nr = __builtin_amdgcn_make_buffer_rsrc((void*)(NORM ? p.norm_w : p.x), 0, K * 4, 0x00020000);
  f32x4 xv[kQ4Turns][2], gw[kQ4Turns][2];
#pragma unroll
  for (int j = 0; j < kQ4Turns; ++j)
    if (j * kQ4Threads * 8 < K) {
      const int k = (tid + j * kQ4Threads) * 8;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        xv[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, k * 4 + 16 * i, 0, 0));
        if (NORM) gw[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(nr, k * 4 + 16 * i, 0, 0));
      }
    }
  __builtin_amdgcn_sched_barrier(0);
  request(0);
  __builtin_amdgcn_sched_barrier(0);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kQ4Turns; ++j)
    if (j * kQ4Threads * 8 < K) {
#pragma clang fp contract(off)      // lo is the split of the ROUNDED product
      const int k8 = tid + j * kQ4Threads;
      bf16x8_t hi, lo;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (NORM) ss = sumsq4(ss, xv[j][i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int kk = (e >> 1) + (e & 1) * 4;                           // places 0 .. 7 hold k = 0 4 1 5 2 6 3 7
        float v = xv[j][kk >> 2][kk & 3];
        if (NORM) v *= gw[j][kk >> 2][kk & 3];
        const __bf16 h = (__bf16)v;
        hi[e] = h;
        lo[e] = (__bf16)(v - (float)h);
      }
      const int at = (k8 >> 6) * 4 + (k8 & 3), pp = (k8 >> 2) & 15;      // unit and eight of 32 codes, place of the 32 (part pp >> 2, group pp & 3)
      if (k8 < S * 64) {
        char* to = xs + at * kQ4Piece + ((pp & 3) * 8 + (pp >> 2) * 2) * 16;
        *reinterpret_cast<bf16x8_t*>(to) = hi;
        *reinterpret_cast<bf16x8_t*>(to + 16) = lo;
      }
    }
  if (NORM) {                              // the factor 1 / rms is applied to the sums: x need not wait for it
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
  }
#pragma unroll
  for (int b = 1; b < kQ4Ahead; ++b) request(b);
  __syncthreads();

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int col = lane & 15;
  bool finite = true;                                                    // of all sums so far
  auto flush = [&]() __attribute__((always_inline)) {                    // rows 4 kq .. of the product belong to part kq: columns 2 kq and 2 kq + 1 are theirs
    if ((col >> 1) == kq) part[(q * kQ4Waves + wave) * 8 + col] = acc;
#pragma unroll
    for (int j = 0; j < 4; ++j) finite &= __builtin_isfinite(acc[j]);
    acc = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  auto unit = [&](int b, auto plain_c) __attribute__((always_inline)) {
    constexpr bool PLAIN = decltype(plain_c)::value;                     // the code itself times the scale: two operations more a code, no scale * 2^24
    const char* xp = xs + s * 4 * kQ4Piece + (kq * 8 + (lane & 7)) * 16;
    const float sc = __uint_as_float(zv[b].x), sc0 = PLAIN ? sc : sc * 16777216.f, sc4 = PLAIN ? sc : sc0 * 0.0625f, nz = -__uint_as_float(zv[b].y);
    const float c0 = PLAIN ? 16777216.f : 1.f, c4 = PLAIN ? 1048576.f : 1.f;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t v = cv[b][m], u = v >> 8;
      const f16x2_t h[4] = {__builtin_bit_cast(f16x2_t, v & 0x000f000fu), __builtin_bit_cast(f16x2_t, v & 0x00f000f0u), __builtin_bit_cast(f16x2_t, u & 0x000f000fu),
                            __builtin_bit_cast(f16x2_t, u & 0x00f000f0u)};
      bf16x8_t w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[2 * e] = (__bf16)fmaf((float)h[e].x * (e & 1 ? c4 : c0), e & 1 ? sc4 : sc0, nz);
        w[2 * e + 1] = (__bf16)fmaf((float)h[e].y * (e & 1 ? c4 : c0), e & 1 ? sc4 : sc0, nz);
      }
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, *reinterpret_cast<const bf16x8_t*>(xp + m * kQ4Piece), acc, 0, 0, 0);
    }
    if (++s == S) { flush(); s = 0; ++q; }
  };
  // (one loop, compact: a launch pays for every line of code it touches; what lies past the end is skipped, its requests return nothing)
  for (int t = 0; t < cnt; t += kQ4Bufs) {
#pragma unroll
    for (int b = 0; b < kQ4Bufs; ++b) {
      request((b + kQ4Ahead) % kQ4Bufs);
      __builtin_amdgcn_sched_barrier(0);
      if (t + b < cnt) unit(b, std::false_type{});
    }
  }
  if (cnt > 0 && s > 0) flush();
  if (__ballot(!finite)) {                 // scale * 2^24 overflows from 2^104 on, and its products are infinite or NaN: this wave's share once more, code by code
    rq = q = first_q; rs = s = i0 - first_q * S; ri = 0;
#pragma unroll 1
    for (int t = 0; t < cnt; ++t) {
      request(0);
      unit(0, std::true_type{});
    }
    if (cnt > 0 && s > 0) flush();
  }
  __syncthreads();

  q4_finish<EPI, NORM, kQ4Waves>(p, part, red, tid, q0, nq, S, items);
#endif
}

template <int EPI, bool NORM>
static int launch4_t(const Gemv4Params& p, int grid, size_t lds, hipStream_t s) {
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv4_kernel<EPI, NORM>), hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemv4: cannot reserve 156 KB of LDS: %s", hipGetErrorString(e));
    configured = true;
  }
  hipLaunchKernelGGL((gemv4_kernel<EPI, NORM>), dim3(grid), dim3(64 * kQ4Waves), lds, s, p);
  CHATTS_CHECK_LAUNCH("gemv4");
  return CHATTS_OK;
}
template <int EPI>
static int launch4_e(const Gemv4Params& p, int grid, size_t lds, hipStream_t s) {
  return p.norm_w ? launch4_t<EPI, true>(p, grid, lds, s) : launch4_t<EPI, false>(p, grid, lds, s);
}

// Which 4-bit projections run here: 16-byte pieces of a row (ldw4 and the pointer in 16 bytes), groups of at least the 32 codes of a lane, x in four turns of a
// workgroup and everything in LDS.  The rest keeps gemv4_ldsx_kernel.  *done: whether this call launched.
int launch_gemv4(const ChattsLinearArgs* a, hipStream_t s, bool* done) {
  Gemv4Params p;
  p.w4 = a->w4; p.sz = reinterpret_cast<const float2*>(a->w4_sz); p.x = a->a; p.norm_w = a->norm_w; p.bias = a->bias; p.resid = a->resid; p.out = a->c; p.eps = a->norm_eps;
  p.n = a->n; p.k = a->k; p.ldw4 = a->ldw4; p.ng = a->k / a->w4_group; p.gshift = 31 - __builtin_clz(a->w4_group);
  const int quads = a->n / 4, cus = device_cus(), grid = quads < cus ? quads : cus, parts = q4_parts(a->k);
  p.quads_each = quads / grid; p.quads_more = quads % grid;
  p.parts_inv = parts > 1 ? (unsigned)((0x100000000ull + parts - 1) / parts) : 0u;      // (units of a workgroup stay below 65536)
  const size_t lds = q4_lds(a->k, (quads + grid - 1) / grid, kQ4Waves);
  // Short rows of few codes stay with gemv4_ldsx_kernel: laying x out as operands and the reduction over the waves cost 4.3 us before any code is read, its batches
  // 3 us and a step for every 1024 codes a row.  us there / here: 1024 x 512 3.0 / 4.3, 4096 x 1024 3.8 / 4.4, 8192 x 1024 4.55 / 4.8, 6144 x 2048 5.1 / 5.9, 1536 x 2560 4.7 / 5.2,
  // 4096 x 2560 5.2 / 5.45; but 7168 x 1536 1 to 8 % less here, 9728 x 896 6.4 / 5.3, 16384 x 1024 6.5 / 5.6, 3072 x 2560 with the norm 7 % less, and from 3073 codes a row on
  // at any n (1024 x 4096 5.8 / 5.1, 256 x 4096 within 3 %).  Left over: 7168 x 2048 (9 % without the norm), 10240 x 1024 (12 %).
  const bool small = (a->k <= 2048 && (a->n <= 6144 || (size_t)a->n * a->k <= (size_t)1 << 23)) || (a->k <= 3072 && a->n <= (a->norm_w ? 2048 : 4096));
  *done = !small && a->w4_group >= 32 && a->n % 16 == 0 && a->k % 32 == 0 && a->k <= kQ4Turns * kQ4Threads * 8 && a->ldw4 % 16 == 0 && ((uintptr_t)a->w4 % 16) == 0 && ((uintptr_t)a->a % 16) == 0 &&
          ((uintptr_t)a->norm_w % 16) == 0 && (size_t)a->n * a->ldw4 < kQ4Far && (size_t)a->n * p.ng * 8 < kQ4Far && ((uintptr_t)a->w4_sz % 8) == 0 && lds <= 156 * 1024 &&
          (a->epilogue == CHATTS_EPI_NONE || a->epilogue == CHATTS_EPI_RESID || a->epilogue == CHATTS_EPI_SWIGLU);
  if (!*done) return CHATTS_OK;
  switch (a->epilogue) {
    case CHATTS_EPI_RESID: return launch4_e<CHATTS_EPI_RESID>(p, grid, lds, s);
    case CHATTS_EPI_SWIGLU: return launch4_e<CHATTS_EPI_SWIGLU>(p, grid, lds, s);
    default: return launch4_e<CHATTS_EPI_NONE>(p, grid, lds, s);
  }
}

}  // namespace chatts
