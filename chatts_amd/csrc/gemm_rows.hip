// gemm_rows.hip - projections of 2 .. 8 rows (decoding for a few sequences at once) without a split of K over workgroups.
//
// What bounds such a projection: W is read once from HBM, and everything else is fixed cost.  gemm_stream_kernel's 128-column tiles need K split
// over workgroups to fill the chip, so every projection drags a second launch behind it that sums the slabs (three in a layer of 110 us), and a barrier per K-step couples all waves of a workgroup to the slowest load.  Here every workgroup owns a few columns for the
// WHOLE of K:
//   * the output columns are dealt to one workgroup per CU in groups of 4 (gated units: 4 gates + their 4 up rows), so 5120 columns are 20 per
//     workgroup on all 256 CUs instead of 40 tiles;
//   * its waves take the K ranges that gemm_stream_kernel gives to its splits.  Each streams its own pieces of W (8 rows x one 128-byte line,
//     LDS-DMA) through a private ring and keeps its X fragments in registers: no barrier before the last K-step, every wave waits for its own loads;
//   * loads run LA K-steps ahead.  Requests past the end of a wave's range carry an offset outside the buffer's bounds: they return nothing and
//     cost nothing, and the counted waits stay constants;
//   * the partial sums meet in LDS and the epilogue (scale, bias, activation, residual, planes) runs once, in the same launch.
// A sum sees the same products in the same order as gemm_stream_kernel's split and its epilogue give it: bit-identical, so the choice between the
// two may depend on the number of rows.  The price is that every workgroup reads all of X from L2 (M x K x 4 bytes instead of a K-range of it).
//
// RMSNorm across the launch: the columns of a row lie in all workgroups, so the projection that updates the residual stream writes
// norm_w * x as planes, WITHOUT the factor 1 / rms, and each workgroup's sum of squares per row (post_ss); the projection that reads these planes
// sums the parts while its first weights travel and multiplies every K range's sums by 1 / rms at the end (row_ss), as gemm_stream_kernel does with what
// goes to its slabs.  Products are linear in the row, so this is the same value with one rounding moved.
#include <type_traits>

#include "gemm_common.h"

namespace chatts {

constexpr int kRowsMaxFN = 4, kRowsRows = 4;         // (8 rows over at least two waves)
// offsets past the end of every buffer the launcher admits: of a K-step, of a row of X that is not there (planes and what lies between them stay below 1 GB; the sum of both does not wrap)
constexpr unsigned kRowsFar = 0x7ffffff0u, kRowsNoToken = 0x40000000u;

// LDS of one wave: LA + 1 K-steps of NP pieces, and 1 KB that the reads of a half fragment may run into
constexpr int rows_ring(int np, int la) { return (la + 1) * np * 1024 + 1024; }

template <bool W8, bool I8, int NP, int LA, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void gemm_rows_kernel(GemmParams p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, int groups_each, int groups_more) {
#ifdef __HIP_DEVICE_COMPILE__      // (buffer resources are a type of the device pass)
  constexpr int FN = (NP + 1) / 2, BK = W8 ? 128 : 64, KS = BK / 32, NX = KS, NB = LA + 1;
  constexpr int RING = rows_ring(NP, LA);
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ float rstd_s[16];
  __shared__ float ss_s[kRowsMaxFN][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool glu = epi_is_glu(p.epilogue);
  const int b0 = (int)blockIdx.x, more = b0 < groups_more;
  const int rows = (groups_each + more) * 4, r0 = (b0 * groups_each + (more ? b0 : groups_more)) * 4;      // columns of this workgroup (gated: gates), the first of them
  constexpr int FG = FN > 1 ? FN / 2 : 1;              // gated: fragments 0 .. FG - 1 are gates, the others their up rows

  // rows of W behind logical row i of fragment f (rows past the end repeat the last one; their sums are dropped)
  auto row_of = [&](int f, int i) __attribute__((always_inline)) {
    if (glu) {
      int at = (f % FG) * 16 + i;
      at = r0 + (at < rows ? at : rows - 1);
      return (at >> 4) * 32 + (at & 15) + (f >= FG ? 16 : 0);
    }
    const int at = f * 16 + i;
    return r0 + (at < rows ? at : rows - 1);
  };

  const int waves = blockDim.x >> 6, nu = p.k / BK, ups = p.k_per_split / BK, kwaves = (nu + ups - 1) / ups, u0 = wave * ups;
  int cnt = ups < nu - u0 ? ups : nu - u0;
  if (cnt < 0) cnt = 0;                                // (a wave more than K ranges: it only helps to finish)
  const unsigned wbytes = W8 ? (unsigned)p.n * (unsigned)p.ldw8 : (unsigned)p.n * (unsigned)p.ldw * 2u;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(W8 ? (void*)p.w8 : (void*)p.w, 0, (int)wbytes, 0x00020000);
  // byte offsets of this lane: of its 16 bytes of every piece (chunk c of row r lies at c ^ ((r >> 1) & 7), applied on the source side), and of its X chunk
  unsigned woff[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const int i = (q & 1) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((i >> 1) & 7);
    woff[q] = (unsigned)row_of(q >> 1, i) * (unsigned)(W8 ? p.ldw8 : 2 * p.ldw) + (unsigned)(u0 * 128 + chunk * 16);
  }
  // X: one load holds both planes of the (at most 8) rows - lanes 0 .. 7 of a 16-lane row the hi plane's, 8 .. 15 the lo plane's - as the columns of the
  // hi product; rotated by 8 lanes it is the lo product's operand.  The other eight columns of either product are sums that nothing reads.
  const int tok = lane & 15, kq = lane >> 4;
  const ptrdiff_t apart = reinterpret_cast<const char*>(a_lo) - reinterpret_cast<const char*>(a_hi);
  const uint16_t* xbase = apart < 0 ? a_lo : a_hi;      // one resource that spans both planes (the launcher has checked how far apart they are)
  const unsigned far = (unsigned)(apart < 0 ? -apart : apart), span = (unsigned)p.m * (unsigned)ldp * 2u;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)xbase, 0, (int)(far + span), 0x00020000);
  const int xrow = tok & 7, second = (tok >> 3) != (apart < 0);
  const unsigned xoff = xrow < p.m ? (second ? far : 0u) + (unsigned)xrow * (unsigned)ldp * 2u + (unsigned)(u0 * BK * 2 + kq * 16) : kRowsNoToken;
  char* ring = smem + wave * RING;

  u32x4 x[NB][KS];
  auto request = [&](int u, int b) __attribute__((always_inline)) {       // K-step u of this wave -> registers b, ring slot b
    __builtin_amdgcn_sched_barrier(0);
    const unsigned xk = u < cnt ? (unsigned)u * (BK * 2) : kRowsFar, wk = u < cnt ? (unsigned)u * 128u : kRowsFar;
#pragma unroll
    for (int h = 0; h < KS; ++h) x[b][h] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff + xk + h * 64, 0, 0);
#pragma unroll
    for (int q = 0; q < NP; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lptr_t)(ring + (b * NP + q) * 1024), 16, woff[q] + wk, 0, 0, 2 /* nt: streamed once */);
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4 acc[FN];
  f32x4 rs_part[kRowsRows];
#pragma unroll
  for (int f = 0; f < FN; ++f) acc[f] = (f32x4){0.f, 0.f, 0.f, 0.f};
  row_rstd_load(p, wave, waves, lane, rs_part);   // (used at the very end)
#pragma unroll
  for (int i = 0; i < LA; ++i) request(i, i);

  auto step = [&](int b) __attribute__((always_inline)) {
    const char* base = ring + b * NP * 1024;
    bf16x8_t wf[FN][KS];
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
      for (int h = 0; h < KS; ++h) {
        const int r = lane & 15;
        if (W8) {                                      // 8 weights = 8 bytes at byte 32 h + 8 kq of the line
          const int c = (2 * h + (kq >> 1)) ^ ((r >> 1) & 7);
          const u32x2 q8 = *reinterpret_cast<const u32x2*>(base + f * 2048 + r * 128 + (c << 4) + (kq & 1) * 8);
          wf[f][h] = I8 ? widen_i8(q8) : widen_fp8(q8);
        } else {
          const int c = (4 * h + kq) ^ ((r >> 1) & 7);
          wf[f][h] = *reinterpret_cast<const bf16x8_t*>(base + f * 2048 + r * 128 + (c << 4));
        }
      }
#pragma unroll
    for (int h = 0; h < KS; ++h) {
      u32x4 turned;
#pragma unroll
      for (int j = 0; j < 4; ++j) turned[j] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x[b][h][j], 0x128 /* row_ror:8 */, 0xf, 0xf, false);
      const bf16x8_t l = __builtin_bit_cast(bf16x8_t, turned), hgh = __builtin_bit_cast(bf16x8_t, x[b][h]);
#pragma unroll
      for (int f = 0; f < FN; ++f) acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f][h], l, acc[f], 0, 0, 0);
#pragma unroll
      for (int f = 0; f < FN; ++f) acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f][h], hgh, acc[f], 0, 0, 0);
    }
  };
  // whole turns of the ring, each step with its request LA ahead, then what is left: all of it has been requested
  const int turns = cnt / NB, left = cnt - turns * NB;
  for (int t = 0; t < turns; ++t) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      request(t * NB + b + LA, (b + LA) % NB);         // into the slot that the step before read: its reads have returned, its products used them
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LA * (NX + NP)) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      step(b);
    }
  }
  auto rest = [&](auto self, auto bc) __attribute__((always_inline)) -> void {
    constexpr int b = decltype(bc)::value;
    if constexpr (b < LA) {
      if (b < left) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((LA - 1 - b) * (NX + NP)) : "memory");
        step(b);
        self(self, std::integral_constant<int, b + 1>{});
      }
    }
  };
  rest(rest, std::integral_constant<int, 0>{});
  // wave f finishes fragment f (gated: its gates and their up rows): a lane has rows i0 .. i0 + 3 of token tok.  What the epilogue reads is requested before
  // the waves meet.
  const int f = wave, i0 = f * 16 + kq * 4, col = r0 + i0, nf = glu ? FG : FN;
  const bool live = f < nf && i0 < rows && tok < p.m;
  const int row = live ? row_of(f, kq * 4) : 0;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 sc = zero, scu = zero, bi = zero, biu = zero, rs = zero, pw = zero;
  if (live) {
    if (W8) sc = *reinterpret_cast<const f32x4*>(p.w8_scale + row);
    if (W8 && glu) scu = *reinterpret_cast<const f32x4*>(p.w8_scale + row + 16);
    if (p.bias) bi = *reinterpret_cast<const f32x4*>(p.bias + row);
    if (p.bias && glu) biu = *reinterpret_cast<const f32x4*>(p.bias + row + 16);
    if (p.epilogue == CHATTS_EPI_RESID) rs = *reinterpret_cast<const f32x4*>(p.resid + (size_t)tok * p.ldc + col);
    if (p.post_ss) pw = *reinterpret_cast<const f32x4*>(p.post_w + col);
  }
  row_rstd_store(p, wave, waves, lane, rs_part, rstd_s);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // (requests past the end of a range, too: the partial sums take their place in LDS)
  __syncthreads();
  f32x4* part = reinterpret_cast<f32x4*>(smem);        // [wave][fragment][lane]
  if (p.row_ss) {                                      // (each range's sum, as gemm_stream_kernel's slabs have it; columns 8 .. 15 are nobody's)
    const float inv = rstd_s[xrow];
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[j] *= inv;
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) part[(wave * FN + j) * 64 + lane] = acc[j];
  __syncthreads();
  float ss = 0.f;
  if (live) {
    auto total = [&](int frag, f32x4 scale, f32x4 bias) __attribute__((always_inline)) {      // the waves' sums in wave order, scale and bias
      f32x4 s = part[frag * 64 + lane];
#pragma unroll
      for (int w = 1; w < MAXW; ++w)
        if (w < kwaves) s += part[(w * FN + frag) * 64 + lane];
      if (W8) s *= scale;
      if (p.bias) s += bias;
      return s;
    };
    f32x4 v = total(f, sc, bi);
    if (glu) {
      const f32x4 up = total(f + FG < FN ? f + FG : f, scu, biu);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = glu_value(p.epilogue, v[j], up[j], p.glu_limit, p.glu_alpha);
    } else if (p.epilogue == CHATTS_EPI_GELU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = gelu_erf_f(v[j]);
    } else if (p.epilogue == CHATTS_EPI_RELU2) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = relu2_f(v[j]);
    } else if (p.epilogue == CHATTS_EPI_RESID) {
      v = rs + v;
    }
    if (p.c_hi) store_planes4(p.c_hi + (size_t)tok * p.ldcp + col, p.c_lo + (size_t)tok * p.ldcp + col, v);
    else *reinterpret_cast<f32x4*>(p.c + (size_t)tok * p.ldc + col) = v;
    if (p.post_ss) {
      ss = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
      store_planes4(p.post_hi + (size_t)tok * p.ld_post + col, p.post_lo + (size_t)tok * p.ld_post + col, pw * v);
    }
  }
  if (p.post_ss) {                                     // (uniform)
    if (f < FN) {
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      if (lane < 16) ss_s[f][lane] = ss;
    }
    __syncthreads();
    if (tid < 16) {
      float s = ss_s[0][tid];
#pragma unroll
      for (int j = 1; j < FN; ++j) s += ss_s[j][tid];
      p.post_ss[tid * kSsStride + blockIdx.x] = s;
    }
  }
#endif
}

// ---- host side ----------------------------------------------------------------------------------------------------------------------------
int rows_grid(int n, int epilogue) {
  const int groups = n / (epi_is_glu(epilogue) ? 8 : 4), cus = device_cus();
  return groups < cus ? groups : cus;
}
static int rows_pieces(int n, int epilogue) {          // 8-row pieces of a K-step of the largest workgroup
  const bool glu = epi_is_glu(epilogue);
  const int groups = n / (glu ? 8 : 4), grid = rows_grid(n, epilogue), rows = (groups + grid - 1) / grid * 4;
  return glu ? 2 * ((rows + 15) / 16 * 2) : (rows + 7) / 8;
}

static size_t rows_lds(int np, int la, int waves) {
  const size_t rings = (size_t)waves * rows_ring(np, la), sums = (size_t)waves * ((np + 1) / 2) * 1024;
  return rings > sums ? rings : sums;
}
static int rows_waves(int np, int sk) { return sk > (np + 1) / 2 ? sk : (np + 1) / 2; }
// K-steps ahead: ~16 KB a step of a workgroup, five of them in flight cover the latency; 8-bit weights have twice the X registers a step
static int rows_ahead(bool w8, int np, int waves) { return waves > 8 ? 3 : (w8 ? (np > 6 ? 3 : 4) : 5); }

// Is the launch that the split's epilogue costs worth more than X read by every workgroup (M x K x 4 bytes at ~55 KB a us and CU; the split reads a K range of it)?
// Both sides measured back to back in a graph, 380 shapes N 1024 .. 10240, K 2048 .. 16384, residual epilogue, us split / here:
//   * X up to 168 KB where K has five to eight ranges: 4096 x 4096 bf16, 8 rows 10.7 / 9.6; 5120 x 5120, 6 rows 13.0 / 12.5; but 4096 x 12288, 8 rows 20.1 / 23.5;
//   * up to 256 KB with four ranges or fewer, whose split reads a larger part of X itself: 8192 x 8192, 8 rows 32.9 / 31.2; int8 7168 x 11264, 4 rows 18 % less here;
//   * fp8 128 KB with eight ranges, 72 KB with five to seven: 4096 x 9216, 3 rows 13 % less; 4096 x 12288, 4 / 8 rows 13.1 / 13.8 and 13.2 / 17.7; 6144 x 4096, 4 rows
//     13 % less, 6144 x 10240 15 % more.  Its waves spend their time widening W: five to seven waves load the four SIMDs unevenly;
//   * and 8-bit not at all with five to seven ranges where more than a third of the fragments is rows that are not there: fp8 5120 x 13824, 2 rows 15.6 / 17.2;
//   * rows of W 32 KB apart: 4096 x 16384 bf16, 2 rows 33.3 / 37.6;
//   * with more than eight ranges (bf16, up to 2048 columns: more than eight sums to add and eight rows of W or fewer a workgroup), against the epilogue that asks for sixteen slabs at once:
//     72 KB up to twelve ranges (512 x 2304, 8 rows 6.2 / 5.8; 1024 x 3072, 6 / 8 rows 6.4 / 6.4, 6.4 / 7.1); with thirteen and fourteen 36 KB, 72 from 6 million weights on (1024 x 3584, 2 / 4
//     rows 6.3 / 6.3, 6.5 / 6.8; 2048 x 3584, 5 / 7 rows 7.3 / 7.1, 7.5 / 7.8); with more 96 KB from 8 million on (2048 x 6144, 4 / 8 rows 8.9 / 8.5, 9.1 / 10.7; 2048 x 4096, 4 / 8 rows 7.7 / 7.7,
//     7.9 / 8.7) and not below (1024 x 4096, 2 / 8 rows 6.3 / 6.8, 6.6 / 8.4).
//     A norm is handed on from here only (that epilogue does not): 192 KB where one is, against a launch more;
//   * always where the split has more workgroups than CUs: 7168 x 5120 20.6 / 15.7.
// Beyond the line it would still win up to 14 % at K = 8192 with 5 to 8 rows and up to 11 % at 5120 or 6144 columns with K of 9216 to 12288; within it, it loses up to 3 %
// at a few (5120 x 5120, 8 rows; fp8 4096 x 10240, 3 rows: 5 %).
static bool rows_pay(const ChattsLinearArgs* a, int sk, int np, bool hands_on) {
  const int groups = a->n / (epi_is_glu(a->epilogue) ? 8 : 4), grid = rows_grid(a->n, a->epilogue), wrows = (groups + grid - 1) / grid * (epi_is_glu(a->epilogue) ? 8 : 4);
  const bool w8 = a->w8 != nullptr, fp8 = w8 && a->w8_format != CHATTS_W8_INT8;
  if ((a->n + 127) / 128 * sk > device_cus()) return true;
  if (sk > 8) {
    const size_t weights = (size_t)a->n * a->k;
    const int most = hands_on ? 192 : sk <= 12 ? 72 : (sk <= 14 ? (weights >= 6000000 ? 72 : 36) : (weights >= 8000000 ? 96 : 0));
    return (size_t)a->m * a->k * 4 <= (size_t)most * 1024;
  }
  if (sk > 4 && (w8 ? (size_t)a->ldw8 : 2 * (size_t)a->ldw) >= 32768) return false;
  if (sk > 4 && sk < 8 && w8 && 16 * ((np + 1) / 2) * 2 > 3 * wrows) return false;
  const int kb = sk <= 4 ? 256 : (!fp8 ? 168 : (sk == 8 ? 128 : 72));
  return (size_t)a->m * a->k * 4 <= (size_t)kb * 1024;
}

bool use_rows(const ChattsLinearArgs* a, int sk, bool hands_on) {
  // a workgroup stores its result while others still read A (the split's epilogue is a launch behind them)
  for (int i = 0; i < 3; ++i)
    if (meets_planes(a, result_range(a, i))) return false;
  auto al = [](const void* q) { return ((uintptr_t)q % 16) == 0; };
  const bool w8 = a->w8 != nullptr;
  const size_t wbytes = w8 ? (size_t)a->n * a->ldw8 : (size_t)a->n * a->ldw * 2;
  const int np = rows_pieces(a->n, a->epilogue), waves = rows_waves(np, sk);
  const ptrdiff_t apart = reinterpret_cast<const char*>(a->a_lo) - reinterpret_cast<const char*>(a->a_hi);
  return a->m >= 2 && a->m <= 8 && a->n % 16 == 0 && rows_pay(a, sk, np, hands_on) && !a->planes_tiled && np <= (w8 ? 2 * kRowsMaxFN : 6) && waves <= (np == 1 && !w8 ? 16 : 8) && (!w8 || a->m <= 4 || waves == 8) &&
         rows_lds(np, rows_ahead(w8, np, waves), waves) <= 156 * 1024 && wbytes < kRowsFar && (size_t)(apart < 0 ? -apart : apart) + (size_t)a->m * a->ld_planes * 2 < kRowsNoToken && a->ldc % 4 == 0 &&
         al(a->c) && al(a->resid) && al(a->bias) && al(a->w8_scale) &&
         (!a->c_hi || (a->ld_cplanes % 4 == 0 && ((uintptr_t)a->c_hi % 8) == 0 && ((uintptr_t)a->c_lo % 8) == 0));
}

template <bool W8, bool I8, int NP, int LA, int MAXW = 8>
static int launch_rows_t(const GemmParams& p, const ChattsLinearArgs* a, int waves, hipStream_t s) {
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_rows_kernel<W8, I8, NP, LA, MAXW>), hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemm_rows: cannot reserve 156 KB of LDS: %s", hipGetErrorString(e));
    configured = true;
  }
  const int groups = a->n / (epi_is_glu(a->epilogue) ? 8 : 4), grid = rows_grid(a->n, a->epilogue);
  hipLaunchKernelGGL((gemm_rows_kernel<W8, I8, NP, LA, MAXW>), dim3(grid), dim3(64 * waves), rows_lds(NP, LA, waves), s, p, a->a_hi, a->a_lo, a->ld_planes, groups / grid,
                     groups % grid);
  CHATTS_CHECK_LAUNCH("gemm_rows");
  return CHATTS_OK;
}
template <bool W8, bool I8>
static int launch_rows_w(const GemmParams& p, const ChattsLinearArgs* a, int sk, hipStream_t s) {
  const int np = rows_pieces(a->n, a->epilogue), waves = rows_waves(np, sk);
  constexpr int LA = W8 ? 4 : 5;                       // rows_ahead()
  switch (np) {
    case 1:
      if constexpr (!W8)
        if (waves > 8) return launch_rows_t<false, false, 1, 3, 16>(p, a, waves, s);
      return launch_rows_t<W8, I8, 1, LA>(p, a, waves, s);
    case 2: return launch_rows_t<W8, I8, 2, LA>(p, a, waves, s);
    case 3: return launch_rows_t<W8, I8, 3, LA>(p, a, waves, s);
    case 4: return launch_rows_t<W8, I8, 4, LA>(p, a, waves, s);
    case 5: return launch_rows_t<W8, I8, 5, LA>(p, a, waves, s);
    case 6: return launch_rows_t<W8, I8, 6, LA>(p, a, waves, s);
    default:                                           // (bf16: use_rows has refused)
      if constexpr (W8) return np == 7 ? launch_rows_t<true, I8, 7, 3>(p, a, waves, s) : launch_rows_t<true, I8, 8, 3>(p, a, waves, s);
      return CHATTS_E_SHAPE;
  }
}
int launch_rows(const GemmParams& p, const ChattsLinearArgs* a, int sk, hipStream_t s) {
  if (!a->w8) return launch_rows_w<false, false>(p, a, sk, s);
  return a->w8_format == CHATTS_W8_INT8 ? launch_rows_w<true, true>(p, a, sk, s) : launch_rows_w<true, false>(p, a, sk, s);
}

}  // namespace chatts
