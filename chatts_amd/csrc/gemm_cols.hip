// gemm_cols.hip - wide projections of 2 .. 16 rows (gate_up, the vocabulary projection of a batched step): every workgroup owns a share of the columns for the whole of K.
//
// What bounds such a projection: W is read once from HBM.  gemm_stream_kernel left three things on the table: 128-column tiles are 192 or 216 workgroups on 256 CUs (or half of
// that twice over, with slabs and a second launch behind them), a barrier per K-step ties all waves to the slowest load, and all workgroups walk K in step - rows 8 KB apart then
// ask the same memory channels and banks at the same time (24576 x 4096 took 1.2 times as long per byte as the same matrix with rows 256 bytes further apart).  Here:
//   * the columns are dealt to one workgroup per CU in groups of 4 (gated units: 4 gates + their 4 up rows), in panels of at most 128 rows of W;
//   * its waves share K: each has a range of its own, streams its pieces of W (8 rows x one 128-byte line, LDS-DMA) through a private ring, a fragment of 16 rows at a time, and meets
//     the other waves only behind the last K-step of a panel.  The next panel's first pieces are under way by then;
//   * a workgroup starts at a hashed K-step of each range and goes round: at any time the card reads all places of a row;
//   * X comes through LDS, too (8 rows x 128 bytes a piece): read as fragments from memory, 16 rows x 64 bytes, it took as long as W at 16 rows of 8-bit weights.
// Neither more in flight (8 fragments ahead instead of 4 .. 6) nor 256-byte pieces changed anything; four waves with deep rings beat eight with shallow ones from 96 rows on
// (32.6 / 35.1 us), below that eight keep enough in flight.  Measured in a graph over rotating weights, gemm_stream_kernel / here, us:
//   24576 x 4096 gated bf16: 5 rows 39 / 32.5, 16 rows 40.7 / 33.0 (6.1 TB/s); fp8 25.8 / 20.9;   27648 x 5120 gated: fp8 5 / 16 rows 28.1 / 27.5, 31.2 / 30.3, bf16 47.4 / 45.7, 49.3 / 47.4
//   151936 x 4096 bf16: 236 / 189, 242 / 204;   152064 x 5120 fp8: 134 / 124, 153 / 145;   32000 x 2048 bf16: 31 / 23.7
// A column's sum runs over the K ranges' sums in wave order, each from its hashed start on, the lo product before the hi one: N, the epilogue and the weight format decide it, the
// number of rows does not.
#include <type_traits>

#include "gemm_common.h"

namespace chatts {

// an offset past the end of every buffer that the launcher admits (two of them do not wrap)
constexpr unsigned kColsFar = 0x7ffffff0u;

constexpr int kColsTurns = 4;         // columns (gates and up rows) of a workgroup: at most so many a thread

// (8-bit weights keep four waves: X of a K-step is twice as large)
constexpr int cols_waves(bool w8, int fn) { return !w8 && fn == 4 ? 8 : 4; }
constexpr int cols_x_pieces(bool w8, bool m8) { return (w8 ? 8 : 4) / (m8 ? 2 : 1); }      // X of a K-step: (plane, 64 k) x 8 rows
// fragments of W that are requested before the one that is read; 1 KB pieces of a wave: X of two K-steps, those fragments and that one
constexpr int cols_ahead(int fn) { return fn == 4 ? 4 : fn - 2; }
constexpr int cols_ring(bool w8, bool m8, int fn) { return 2 * cols_x_pieces(w8, m8) + 2 * (cols_ahead(fn) + 1); }
// the place of chunk c of row r: ds_read_b128 / b64 of 16 rows at once meet no bank twice
__device__ __forceinline__ int cols_swizzle(int r) { return (r >> 1) & 7; }

struct ColsGeom {
  int groups_each, groups_more;      // groups of 4 columns of a workgroup; the first groups_more workgroups have one more
  int panels;                        // a workgroup walks its columns in this many panels
  int sums_at, scale_at, bias_at;    // LDS offsets
};

// FN: 16-row fragments of a panel (gated: FN / 2 of gates, then those of their up rows).
template <bool W8, bool I8, bool GLU, int FN, bool M8>
__global__ __launch_bounds__(64 * cols_waves(W8, FN)) void gemm_cols_kernel(GemmParams p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, ColsGeom g) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int NW = cols_waves(W8, FN), FG = GLU ? FN / 2 : FN, BK = W8 ? 128 : 64, KS = BK / 32, NSUB = BK / 64, NX = cols_x_pieces(W8, M8), AHEAD = cols_ahead(FN), RS = 2 * (AHEAD + 1);
  constexpr int SUB = M8 ? 1024 : 2048;                // X rows of 64 k: 8 or 16
  static_assert(AHEAD <= FN, "the wait for the first fragment of a K-step stands for its X, too");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ float rstd_s[16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b0 = (int)blockIdx.x, more = b0 < g.groups_more, groups = g.groups_each + more;
  const int r0 = (b0 * g.groups_each + (more ? b0 : g.groups_more)) * 4;      // first column (gated: gate)
  auto panel_from = [&](int j) __attribute__((always_inline)) { return j * groups / g.panels * 4; };      // first column of panel j, from r0

  // this wave's K-steps: u0 .. u0 + cnt - 1, from u0 + first on and round
  const int nk = p.k / BK, u0 = wave * nk / NW, cnt = (wave + 1) * nk / NW - u0;
  const int first = (int)__umulhi((unsigned)b0 * 0x9E3779B1u, (unsigned)cnt);
  const unsigned wbytes = W8 ? (unsigned)p.n * (unsigned)p.ldw8 : (unsigned)p.n * (unsigned)p.ldw * 2u;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(W8 ? (void*)p.w8 : (void*)p.w, 0, (int)wbytes, 0x00020000);
  const unsigned abytes = ((unsigned)(p.m - 1) * (unsigned)ldp + (unsigned)p.k) * 2u;
  const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc((void*)a_hi, 0, (int)abytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t lr = __builtin_amdgcn_make_buffer_rsrc((void*)a_lo, 0, (int)abytes, 0x00020000);
  const int tok = lane & 15, kq = lane >> 4;
  char* xring = smem + wave * (cols_ring(W8, M8, FN) * 1024);
  char* ring = xring + 2 * NX * 1024;

  unsigned woff[FN * 2];
  auto place = [&](int panel) __attribute__((always_inline)) {      // this lane's sources in the panel, but for the K-step
    const int c0 = panel_from(panel), rows = panel_from(panel + 1) - c0;
#pragma unroll
    for (int q = 0; q < FN * 2; ++q) {
      const int f = q / 2, half = GLU ? f / FG : 0, i = (q % 2) * 8 + (lane >> 3), at = (f - half * FG) * 16 + i;      // row i of fragment f
      const int col = r0 + c0 + at, row = GLU ? (col >> 4) * 32 + (col & 15) + half * 16 : col;
      const int chunk = (lane & 7) ^ cols_swizzle(i);
      woff[q] = at < rows ? (unsigned)row * (unsigned)(W8 ? p.ldw8 : 2 * p.ldw) + (unsigned)chunk * 16u : kColsFar;
    }
  };
  // the K-step whose pieces are requested next, a fragment at a time, into the two slots of the ring from rslot on
  int ru = u0 + first, rleft = cnt, rp = 0, rslot = 0;
  bool live = cnt > 0;
  auto request = [&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value;
    const unsigned wk = live ? (unsigned)ru * 128u : kColsFar;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const unsigned at = woff[f * 2 + i] + wk;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lptr_t)(ring + (rslot + i) * 1024), 16, at, 0, 0, 2 /* nt: streamed once */);
    }
    __builtin_amdgcn_sched_barrier(0);
    rslot = rslot + 2 == RS ? 0 : rslot + 2;
    if constexpr (f == FN - 1) {
      if (++ru == u0 + cnt) ru = u0;
      if (--rleft == 0) {
        rleft = cnt;
        if (++rp < g.panels) place(rp);
        else live = false;
      }
    }
  };
  // X of a K-step: rows that are not there stay out
  unsigned xoff[NX / 2];
#pragma unroll
  for (int q = 0; q < NX / 2; ++q) {                   // of a plane: (64 k, 8 rows)
    const int sub = M8 ? q : q / 2, r = (M8 ? 0 : q % 2) * 8 + (lane >> 3), chunk = (lane & 7) ^ cols_swizzle(r);
    xoff[q] = r < p.m ? (unsigned)r * (unsigned)ldp * 2u + (unsigned)(sub * 128 + chunk * 16) : kColsFar;
  }
  int xu = u0 + first, xslot = 0;
  auto request_x = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const unsigned k = cnt > 0 ? (unsigned)xu * (BK * 2) : kColsFar;
#pragma unroll
    for (int q = 0; q < NX; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(q < NX / 2 ? hr : lr, (lptr_t)(xring + (xslot * NX + q) * 1024), 16, xoff[q % (NX / 2)] + k, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    xslot ^= 1;
    if (++xu == u0 + cnt) xu = u0;
  };

  f32x4 rs_part[16 / NW];
  // [gate | up] scales and biases of this workgroup's columns: requested first, in LDS when they are needed
  float* scale_s = reinterpret_cast<float*>(smem + g.scale_at);
  float* bias_s = reinterpret_cast<float*>(smem + g.bias_at);
  float sc_r[kColsTurns], bi_r[kColsTurns];
#pragma unroll
  for (int t = 0; t < kColsTurns; ++t) {
    const int i = tid + t * 64 * NW, half = i >= groups * 4, at = r0 + i - half * groups * 4;
    int row = GLU ? (at >> 4) * 32 + (at & 15) + half * 16 : at;
    if (row > p.n - 1) row = p.n - 1;
    if (W8) sc_r[t] = p.w8_scale[row];
    if (p.bias) bi_r[t] = p.bias[row];
  }
  row_rstd_load(p, wave, NW, lane, rs_part);
  place(0);
  request_x();
  auto every = [&](auto self, auto fc) __attribute__((always_inline)) -> void {
    constexpr int f = decltype(fc)::value;
    if constexpr (f < AHEAD) {
      request(fc);
      self(self, std::integral_constant<int, f + 1>{});
    }
  };
  every(every, std::integral_constant<int, 0>{});
  f32x4 acc[FN];
#pragma unroll
  for (int f = 0; f < FN; ++f) acc[f] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int slot = 0, xread = 0;
  const int sw = cols_swizzle(tok);
  bf16x8_t xhi[KS], xlo[KS];
  auto step = [&](auto self, auto fc) __attribute__((always_inline)) -> void {
    constexpr int f = decltype(fc)::value;
    if constexpr (f < FN) {
      // younger than this fragment's pieces: those of the AHEAD - 1 fragments behind it, and the X of the next step where this fragment was requested in the step before
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * 2 + (f < AHEAD ? NX : 0)) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (f == 0) {
#pragma unroll
        for (int h = 0; h < KS; ++h) {
          const char* at = xring + xread * (NX * 1024) + (h >> 1) * SUB + tok * 128 + ((((h & 1) * 4 + kq) ^ sw) << 4);
          xhi[h] = *reinterpret_cast<const bf16x8_t*>(at);
          xlo[h] = *reinterpret_cast<const bf16x8_t*>(at + NSUB * SUB);
        }
        xread ^= 1;
      }
      const char* base = ring + slot * 1024 + tok * 128;
      slot = slot + 2 == RS ? 0 : slot + 2;
      bf16x8_t wf[KS];
#pragma unroll
      for (int h = 0; h < KS; ++h) {
        if (W8) {
          const u32x2 q8 = *reinterpret_cast<const u32x2*>(base + (((2 * h + (kq >> 1)) ^ sw) << 4) + (kq & 1) * 8);
          wf[h] = I8 ? widen_i8(q8) : widen_fp8(q8);
        } else {
          wf[h] = *reinterpret_cast<const bf16x8_t*>(base + (((4 * h + kq) ^ sw) << 4));
        }
      }
      request(std::integral_constant<int, (f + AHEAD) % FN>{});      // into the slots that the fragment before this one was read from
#pragma unroll
      for (int h = 0; h < KS; ++h) {
        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h], xlo[h], acc[f], 0, 0, 0);
        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h], xhi[h], acc[f], 0, 0, 0);
      }
      self(self, std::integral_constant<int, f + 1>{});
    }
  };
  auto finish = [&](int panel) __attribute__((always_inline)) {
    const int c0 = panel_from(panel), rows = panel_from(panel + 1) - c0;
    f32x4* part = reinterpret_cast<f32x4*>(smem + g.sums_at);        // [wave][fragment][lane]
    if (panel == 0) {
      row_rstd_store(p, wave, NW, lane, rs_part, rstd_s);
#pragma unroll
      for (int t = 0; t < kColsTurns; ++t) {
        const int i = tid + t * 64 * NW;
        if (i >= groups * 4 * (GLU ? 2 : 1)) break;
        if (W8) scale_s[i] = sc_r[t];
        if (p.bias) bias_s[i] = bi_r[t];
      }
    } else { __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); }
    if (g.sums_at == 0) {              // in the rings' place
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
#pragma unroll
    for (int f = 0; f < FN; ++f) part[(wave * FN + f) * 64 + lane] = acc[f];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const float rstd = p.row_ss ? rstd_s[tok] : 1.f;
    auto total = [&](int f, int at) __attribute__((always_inline)) {      // at: place in the scales
      f32x4 v = part[f * 64 + lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += part[(w * FN + f) * 64 + lane];
      if (p.row_ss) v *= rstd;
      if (W8) v *= *reinterpret_cast<const f32x4*>(scale_s + at);
      if (p.bias) v += *reinterpret_cast<const f32x4*>(bias_s + at);
      return v;
    };
    for (int f = wave; f < FG; f += NW) {
      const int i0 = f * 16 + kq * 4, at = c0 + i0, col = r0 + at;
      if (i0 < rows && tok < p.m) {
        f32x4 v = total(f, at);
        if constexpr (GLU) {
          const f32x4 u = total(f + FG, groups * 4 + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = glu_value(p.epilogue, v[e], u[e], p.glu_limit, p.glu_alpha);
        } else if (p.epilogue == CHATTS_EPI_GELU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_erf_f(v[e]);
        } else if (p.epilogue == CHATTS_EPI_RELU2) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = relu2_f(v[e]);
        } else if (p.epilogue == CHATTS_EPI_RESID) {
          v = *reinterpret_cast<const f32x4*>(p.resid + (size_t)tok * p.ldc + col) + v;
        }
        if (p.c_hi) store_planes4(p.c_hi + (size_t)tok * p.ldcp + col, p.c_lo + (size_t)tok * p.ldcp + col, v);
        else *reinterpret_cast<f32x4*>(p.c + (size_t)tok * p.ldc + col) = v;
      }
    }
#pragma unroll
    for (int f = 0; f < FN; ++f) acc[f] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  int kt = 0, panel = 0;
  if (cnt > 0) {
    while (true) {
      request_x();                       // of the next step, in the place of the last one's
      step(step, std::integral_constant<int, 0>{});
      if (++kt == cnt) {
        kt = 0;
        finish(panel++);
        if (panel == g.panels) break;
      }
    }
  }
  for (; panel < g.panels; ) finish(panel++);      // (a wave without K-steps)
#endif
}

// ---- host side ----------------------------------------------------------------------------------------------------------------------------
constexpr int kColsMaxFN = 8;
// Which projections run here - by the matrix alone, because a row's bits must not depend on the number of rows.  Measured against the split and gemm_rows_kernel, N 8192 .. 24576,
// K 2048 .. 8192, 2 / 8 / 16 rows, with and without a gate (160 shapes): from 12288 columns on 1.0 .. 1.7 times as fast (18432 x 4096 bf16 44 -> 26 us, 16384 x 8192 fp8 37 -> 28), but
// for 12288 x 4096 bf16 of 2 rows without a gate (4 % slower) and fp8 x 5120 of 16 rows at 14336 .. 16384 (up to 6 %); at 10240 0.83 .. 1.2, at 8192 0.6 .. 1.0: a share is then 40 rows or
// less, and X weighs as much as W.  Short K at the lower end stays with the two others, whose widest instances it is: 12288 x 2048 bf16 (2 rows 10.9 / 11.5 us here, 16 rows 16.1 / 12.4)
// and 8-bit up to 16384 x 4096 (4096: 16.0 / 13.9 and 17.2 / 16.1).
static bool cols_pay(const ChattsLinearArgs* a) { return a->w8 ? a->n >= 12288 && (a->k > 4096 || a->n > 16384) : a->n >= 12288 && (a->k > 2048 || a->n > 12288); }
static int cols_grid(int n, int epilogue) {
  const int groups = n / (epi_is_glu(epilogue) ? 8 : 4), cus = device_cus();
  return groups < cus ? groups : cus;
}
static int cols_most(int n, int epilogue) {            // groups of 4 columns of the largest workgroup
  const int groups = n / (epi_is_glu(epilogue) ? 8 : 4), grid = cols_grid(n, epilogue);
  return (groups + grid - 1) / grid;
}
static int cols_panels(int n, int epilogue) {
  const int cap = kColsMaxFN * (epi_is_glu(epilogue) ? 2 : 4);
  return (cols_most(n, epilogue) + cap - 1) / cap;
}
static int cols_fn(int n, int epilogue) {              // 4, 6 or 8 (fragments without rows cost next to nothing)
  const int panels = cols_panels(n, epilogue), rows = (cols_most(n, epilogue) + panels - 1) / panels * 4, fn = (rows + 15) / 16 * (epi_is_glu(epilogue) ? 2 : 1);
  return fn <= 4 ? 4 : (fn <= 6 ? 6 : 8);
}
// dynamic LDS: the rings, behind them (or, for a single panel, in their place) the waves' sums, and the columns' scales and biases.  rstd_s is static beside it
constexpr int kColsLds = 159 * 1024;
static int cols_place(const ChattsLinearArgs* a, bool m8, ColsGeom& g) {
  const bool w8 = a->w8 != nullptr;
  const int fn = cols_fn(a->n, a->epilogue), nw = cols_waves(w8, fn), most = cols_most(a->n, a->epilogue) * (epi_is_glu(a->epilogue) ? 8 : 4) * (int)sizeof(float);
  int at = nw * cols_ring(w8, m8, fn) * 1024;
  g.sums_at = 0;
  if (g.panels > 1) { g.sums_at = at; at += nw * fn * 1024; }
  g.scale_at = at;
  if (w8) at += most;
  g.bias_at = at;
  return a->bias ? at + most : at;
}

bool use_cols(const ChattsLinearArgs* a) {
  const int opt = opt_get(OPT_GEMM_COLS, 1);           // 0: never, 2: wherever it can
  if (opt == 0) return false;
  for (int i = 0; i < 3; ++i)                          // a workgroup stores its result while others still read A
    if (meets_planes(a, result_range(a, i))) return false;
  auto al = [](const void* q, int to) { return ((uintptr_t)q % to) == 0; };
  const bool w8 = a->w8 != nullptr, glu = epi_is_glu(a->epilogue);
  const size_t wbytes = w8 ? (size_t)a->n * a->ldw8 : (size_t)a->n * a->ldw * 2;
  if (!(a->m >= 2 && a->m <= 16 && a->batch <= 1 && a->n % 16 == 0 && (!glu || a->n % 32 == 0) && !a->planes_tiled && wbytes < (size_t)kColsFar &&
        (size_t)a->m * a->ld_planes * 2 < (size_t)kColsFar && cols_most(a->n, a->epilogue) * (glu ? 8 : 4) <= kColsTurns * 256))
    return false;
  ColsGeom g{0, 0, cols_panels(a->n, a->epilogue), 0, 0, 0};
  if (cols_place(a, false, g) > kColsLds) return false;      // (as for 16 rows: the number of rows decides nothing)
  if (a->ldc % 4 != 0 || !al(a->c, 16) || !al(a->resid, 16) || (a->c_hi && (a->ld_cplanes % 4 != 0 || !al(a->c_hi, 8) || !al(a->c_lo, 8)))) return false;
  return opt == 2 || cols_pay(a);
}

template <bool W8, bool I8, bool GLU, int FN, bool M8>
static int launch_cols_t(const GemmParams& p, const ChattsLinearArgs* a, hipStream_t s) {
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_cols_kernel<W8, I8, GLU, FN, M8>), hipFuncAttributeMaxDynamicSharedMemorySize, kColsLds);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemm_cols: cannot reserve %d KB of LDS: %s", kColsLds / 1024, hipGetErrorString(e));
    configured = true;
  }
  constexpr int NW = cols_waves(W8, FN);
  constexpr int ring = NW * cols_ring(W8, M8, FN) * 1024, sums = NW * FN * 1024;
  static_assert(sums <= ring && ring + (FN > 4 ? sums : 0) <= kColsLds && kColsLds + 16 * sizeof(float) <= 160 * 1024, "the sums of a single panel take the rings' place, those of several (of five fragments and more) lie behind them");
  const int groups = a->n / (GLU ? 8 : 4), grid = cols_grid(a->n, a->epilogue);
  ColsGeom g{groups / grid, groups % grid, cols_panels(a->n, a->epilogue), 0, 0, 0};
  const int at = cols_place(a, M8, g);
  hipLaunchKernelGGL((gemm_cols_kernel<W8, I8, GLU, FN, M8>), dim3(grid), dim3(64 * NW), at, s, p, a->a_hi, a->a_lo, a->ld_planes, g);
  CHATTS_CHECK_LAUNCH("gemm_cols");
  return CHATTS_OK;
}
template <bool W8, bool I8, bool M8>
static int launch_cols_w(const GemmParams& p, const ChattsLinearArgs* a, hipStream_t s) {
  const bool glu = epi_is_glu(a->epilogue);
  const int fn = cols_fn(a->n, a->epilogue);
  if (glu) return fn == 4 ? launch_cols_t<W8, I8, true, 4, M8>(p, a, s) : (fn == 6 ? launch_cols_t<W8, I8, true, 6, M8>(p, a, s) : launch_cols_t<W8, I8, true, 8, M8>(p, a, s));
  return fn == 4 ? launch_cols_t<W8, I8, false, 4, M8>(p, a, s) : (fn == 6 ? launch_cols_t<W8, I8, false, 6, M8>(p, a, s) : launch_cols_t<W8, I8, false, 8, M8>(p, a, s));
}
int launch_cols(const GemmParams& p, const ChattsLinearArgs* a, hipStream_t s) {
  const bool m8 = a->m <= 8;
  if (!a->w8) return m8 ? launch_cols_w<false, false, true>(p, a, s) : launch_cols_w<false, false, false>(p, a, s);
  if (a->w8_format == CHATTS_W8_INT8) return m8 ? launch_cols_w<true, true, true>(p, a, s) : launch_cols_w<true, true, false>(p, a, s);
  return m8 ? launch_cols_w<true, false, true>(p, a, s) : launch_cols_w<true, false, false>(p, a, s);
}

}  // namespace chatts
