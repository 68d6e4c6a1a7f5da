// gemv_ring.hip - batch-1 projections of long rows: y[N] = epilogue(W[N,K] . norm(x)), W bf16, fp8 (OCP e4m3fn) or int8 with a power-of-two scale per row.
//
// What bounds it: W is read once from HBM, 6.5 TB/s where enough of it is under way (32 KB a CU) from the launch's start to its end.  gemv_ldsx_kernel (gemv.hip) asks for 2 rows x
// 2 chunks, waits for all of them and computes: 8 waves have 32 KB a CU under way, then nothing, and nothing at all while x is staged.  Here a wave's tasks (two rows each) are
// ONE sequence of units, a 1 KB chunk of each of the task's rows, that runs through a ring of D units in registers: the loads of the next D - 1 units are always under way,
// over the end of a task, too, and the first ones since before x was staged.  Requests past a row's end or the last task lie outside the row's buffer: they return zeros.
// Lane j keeps the j-th task's sums, and the epilogues of up to 64 tasks run side by side behind them: a residual asked for between two units would wait for the whole ring.
// Each row is summed in gemv_ldsx_kernel's order: the same bits, but where a norm is fused: its sum of squares runs over the workgroup's threads, and the two have other numbers of waves.
#include "common.h"
#include "gemv_common.h"

namespace chatts {

constexpr int kFmtBf16 = -1;      // else CHATTS_W8_FP8, CHATTS_W8_INT8

// a lane's own task: all its rows
template <int ROWS, int EPI, bool W8>
__device__ __forceinline__ void gemv_finish(const GemvParams& p, int task, float (&acc)[ROWS]) {
  if constexpr (W8) {                                     // power-of-two scales: exact
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int row = task_row<ROWS, EPI>(task, r);
      acc[r] *= p.w8_scale[row < p.n ? row : 0];
    }
  }
  if constexpr (epi_is_glu(EPI)) {
#pragma unroll
    for (int u = 0; u < ROWS / 2; ++u) {
      const int rg = task_row<ROWS, EPI>(task, 2 * u);
      if (rg + 16 < p.n) p.out[task * (ROWS / 2) + u] = gemv_gated<EPI>(p, rg, acc[2 * u], acc[2 * u + 1]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (task * ROWS + r < p.n) p.out[task * ROWS + r] = gemv_value<EPI>(p, task * ROWS + r, acc[r]);
  }
}

// Rows of a task; units of the ring, two of them under way beside the one that is computed.  More cost code and registers and hide nothing; us with 8 / 6 / 4 / 3 / 2 units: bf16 7168 x 5120
// 14.1 / 13.7 / 13.1 / 13.0 / 13.5, 27648 x 5120 gated 45.3 / 44.9 / 44.7 / 43.9 / 44.5, 4096 x 4096 8.5 / 8.5 / 7.9 / 7.8 / 7.8, 24576 x 4096 gated 32.5 / 32.2 / 32.2 / 31.4 / 31.8, 4096 x 12288
// 18.6 / 18.2 / 18.2 / 18.2 / 18.2; fp8 27648 x 5120 gated 25.4 / 24.9 / 24.2 / 23.5 / 23.9, 5120 x 13824 15.2 / 14.7 / 13.9 / 14.2 / 14.3, 24576 x 4096 gated 18.9 / 18.3 / 17.8 / 17.4 / 17.9.
constexpr int kRingRows = 2, kRingUnits = 3;
constexpr int kGemvTurns = 4;                   // pieces of x that a thread holds while the first weights are requested
template <int EPI, bool NORM, int FMT>
__global__ __launch_bounds__(1024) void gemv_ring_kernel(GemvParams p) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int ROWS = kRingRows, D = kRingUnits;
  constexpr bool W8 = FMT != kFmtBf16;
  constexpr int CE = W8 ? 1024 : 512, CB = W8 ? 10 : 9, Q = CE / 256;      // k of a chunk; x pieces of a lane and chunk
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if (!W8 && gridDim.y > 1) { p.x += blockIdx.y * p.x_stride; p.w += blockIdx.y * p.w_stride; p.out += blockIdx.y * p.out_stride; }
  f32x4* xs4 = reinterpret_cast<f32x4*>(smem);            // permuted x: [chunk][half][lane] float4
  float* red = reinterpret_cast<float*>(smem) + (size_t)((p.k + CE - 1) >> CB) * CE;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nthreads = blockDim.x, nw = nthreads >> 6;
  const int K = p.k;
  const int nchunks = (K + CE - 1) >> CB;
  const int task0 = blockIdx.x * nw + wave, stride = gridDim.x * nw, tasks = task0 < p.tasks ? (p.tasks - 1 - task0) / stride + 1 : 0;

  f32x4 xv[kGemvTurns], gv[kGemvTurns];
#pragma unroll
  for (int j = 0; j < kGemvTurns; ++j) {
    const int k4 = (tid + j * nthreads) * 4;
    xv[j] = gv[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (k4 < K) {
      xv[j] = *reinterpret_cast<const f32x4*>(p.x + k4);
      if (NORM) gv[j] = *reinterpret_cast<const f32x4*>(p.norm_w + k4);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // the unit to request next: chunk rat of task rt, rleft chunks of it to go.  (All rows of a task exist: N is a multiple of 16.)
  u32x4 wv[D][ROWS];
  __amdgpu_buffer_rsrc_t rows[ROWS];
  int rt = task0, rat = 0, rleft = nchunks;
  const size_t ld = W8 ? (size_t)p.ldw8 : (size_t)p.ldw * 2;
  auto place = [&]() __attribute__((always_inline)) {
    const bool live = rt < p.tasks;
    const char* at = (W8 ? reinterpret_cast<const char*>(p.w8) : reinterpret_cast<const char*>(p.w)) + (live ? (size_t)task_row<ROWS, EPI>(rt, 0) * ld : 0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      rows[r] = __builtin_amdgcn_make_buffer_rsrc((void*)(at + (epi_is_glu(EPI) ? (r & 1) * 16 + (r >> 1) : r) * ld), 0, live ? (W8 ? K : 2 * K) : 0, 0x00020000);
    rat = p.spread ? gemv_first_chunk<ROWS>(rt, p.spread) : 0;
  };
  auto request = [&](int b) __attribute__((always_inline)) {
    const unsigned off = (unsigned)rat * 1024u + (unsigned)lane * 16u;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) wv[b][r] = __builtin_amdgcn_raw_buffer_load_b128(rows[r], off, 0, 2 /* nt: streamed once */);
    if (++rat == nchunks) rat = 0;
    if (--rleft == 0) { rleft = nchunks; rt += stride; place(); }
  };
  place();
  constexpr int EARLY = 2;                                // (more would stand in front of the x that later waves ask for)
#pragma unroll
  for (int b = 0; b < EARLY; ++b) request(b);
  __builtin_amdgcn_sched_barrier(0);

  float rstd = 1.f;
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kGemvTurns; ++j)
      if ((tid + j * nthreads) * 4 < K) ss = sumsq4(ss, xv[j]);
    for (int k4 = (tid + kGemvTurns * nthreads) * 4; k4 < K; k4 += nthreads * 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p.x + k4);
      ss = sumsq4(ss, v);
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < nw; ++i) t += red[i];
    rstd = rsqrtf(t / (float)K + p.eps);
  }
  auto stage = [&](int k4, f32x4 v, const f32x4 g) __attribute__((always_inline)) {
    if (NORM) { v.x = g.x * (v.x * rstd); v.y = g.y * (v.y * rstd); v.z = g.z * (v.z * rstd); v.w = g.w * (v.w * rstd); }
    const int chunk = k4 >> CB, within = k4 & (CE - 1);
    if (k4 < nchunks * CE) xs4[(chunk * Q + ((within >> 2) & (Q - 1))) * 64 + within / (4 * Q)] = v;
  };
#pragma unroll
  for (int j = 0; j < kGemvTurns; ++j) stage((tid + j * nthreads) * 4, xv[j], gv[j]);
  for (int k4 = (tid + kGemvTurns * nthreads) * 4; k4 < nchunks * CE; k4 += nthreads * 4) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f}, g = v;
    if (k4 < K) {
      v = *reinterpret_cast<const f32x4*>(p.x + k4);
      if (NORM) g = *reinterpret_cast<const f32x4*>(p.norm_w + k4);
    }
    stage(k4, v, g);
  }
#pragma unroll
  for (int b = EARLY; b < D - 1; ++b) request(b);
  __syncthreads();

  float acc[ROWS], kept[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) { acc[r] = 0.f; kept[r] = 0.f; }
  int task = task0, done = 0, at = p.spread ? gemv_first_chunk<ROWS>(task0, p.spread) : 0, left = nchunks;
  auto unit = [&](int b) __attribute__((always_inline)) {
    f32x4 x[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) x[q] = xs4[(at * Q + q) * 64 + lane];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if constexpr (!W8) acc[r] = dot8(wv[b][r], x[0], x[1], acc[r]);
      else acc[r] = FMT == CHATTS_W8_INT8 ? dot16_i8(wv[b][r], x[0], x[1], x[2], x[3], acc[r]) : dot16_fp8(wv[b][r], x[0], x[1], x[2], x[3], acc[r]);
    }
    if (++at == nchunks) at = 0;
    if (--left == 0) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) acc[r] = wave_sum(acc[r]);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) kept[r] = lane == done ? acc[r] : kept[r];
      ++done;
      left = nchunks;
      task += stride;
      at = p.spread ? gemv_first_chunk<ROWS>(task, p.spread) : 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) acc[r] = 0.f;
    }
  };
  constexpr int BATCH = 64 / D * D;                       // tasks whose sums the lanes keep: whole turns of the ring
  for (int from = 0; from < tasks; from += BATCH) {
    const int some = tasks - from < BATCH ? tasks - from : BATCH, cnt = some * nchunks;
    for (int t = 0; t < cnt; t += D) {
#pragma unroll
      for (int b = 0; b < D; ++b) {
        request((b + D - 1) % D);
        __builtin_amdgcn_sched_barrier(0);
        if (t + b < cnt) unit(b);
      }
    }
    if (lane < some) gemv_finish<ROWS, EPI, W8>(p, task0 + (from + lane) * stride, kept);
    done = 0;
  }
#endif
}

template <int EPI, int FMT>
static void launch_ring_n(const GemvParams& p, bool norm, dim3 grid, int threads, size_t lds, hipStream_t s) {
  if (norm) hipLaunchKernelGGL((gemv_ring_kernel<EPI, true, FMT>), grid, dim3(threads), lds, s, p);
  else hipLaunchKernelGGL((gemv_ring_kernel<EPI, false, FMT>), grid, dim3(threads), lds, s, p);
}
template <int FMT>
static void launch_ring_e(const GemvParams& p, int epi, bool norm, dim3 grid, int threads, size_t lds, hipStream_t s) {
  if (epi == CHATTS_EPI_RESID) return launch_ring_n<CHATTS_EPI_RESID, FMT>(p, norm, grid, threads, lds, s);
  if (epi == CHATTS_EPI_SWIGLU) return launch_ring_n<CHATTS_EPI_SWIGLU, FMT>(p, norm, grid, threads, lds, s);
  if constexpr (FMT == kFmtBf16) {                        // (refused for 8-bit weights)
    if (epi == CHATTS_EPI_RELU2) return launch_ring_n<CHATTS_EPI_RELU2, FMT>(p, norm, grid, threads, lds, s);
    if (epi == CHATTS_EPI_GEGLU) return launch_ring_n<CHATTS_EPI_GEGLU, FMT>(p, norm, grid, threads, lds, s);
    if (epi == CHATTS_EPI_CLAMPGLU) return launch_ring_n<CHATTS_EPI_CLAMPGLU, FMT>(p, norm, grid, threads, lds, s);
  }
  launch_ring_n<CHATTS_EPI_NONE, FMT>(p, norm, grid, threads, lds, s);
}
static size_t ring_lds(const ChattsLinearArgs* a) {
  const int ce = a->w8 ? 1024 : 512;
  return (size_t)((a->k + ce - 1) / ce) * ce * 4 + 64 * 4;
}

// Rows of more than 2048 k: shorter ones are one or two of gemv_ldsx_kernel's batches, and the ring's code costs more than it hides (us there / here: 8192 x 2048 bf16 7.6 / 8.1, fp8
// 5.4 / 6.2; 4096 x 1024 fp8 3.4 / 3.9).  Six tasks a CU: with fewer the K split has more under way.  8-bit weights of more than 32 MB (6144 x 4096 int8 7.5 / 7.9, 5120 x 5120 7.7 / 8.0,
// 8192 x 4096 8.7 / 8.9), and with 9 to 12 tasks a CU, whose waves suit neither one walk nor two, from 44 MB on (fp8 5120 x 8192 10.1 / 10.4, 6144 x 7168 10.8 /
// 11.2, 5120 x 10240 11.6 / 11.4).
// Vocabularies in bf16 (hundreds of tasks a CU) keep two workgroups a CU of that kernel: 152064 x 5120 232 / 235, 151936 x 4096 192 / 192.
// The exchange over ranks stays there, too: its pushes stand between the loads.
bool gemv_ring_takes(const ChattsLinearArgs* a) {
  const int opt = opt_get(OPT_GEMV_RING, 1);              // 0: never, 2: wherever it can
  if (opt == 0 || a->w4 || a->tp_reduce || ring_lds(a) > 64 * 1024 || a->n % 2 != 0) return false;
  const int tasks = a->n / 2, batch = a->batch > 1 ? a->batch : 1;
  const size_t per_cu = (size_t)tasks * batch / device_cus();
  const size_t bytes = (size_t)a->n * a->k, each = (tasks + device_cus() - 1) / device_cus();
  return opt == 2 || (a->k > 2048 && per_cu >= 6 && (a->w8 ? bytes > (size_t)32 << 20 && (each < 9 || each > 12 || bytes >= (size_t)44 << 20) : per_cu < 128));
}

// Waves of a workgroup, one of which a CU has; each keeps 4 KB under way.  Eight of them, or as many as let all walk the same number of tasks where a CU has few: a wave that walks one more
// holds the launch up.  More only stretch the prologue, which long rows bear (7168 x 5120, 14 tasks a CU, 12 / 8 waves 17.1 / 14.2 us, fp8 10.4 / 9.0).  As a part of gemv_ldsx_kernel's time,
// 8 waves / the choice:
//   5 .. 8 tasks: one a wave.
//   9 or 10: 12 for K from 8192 on (4608 x 12288 1.22 / 0.96, fp8 5120 x 12288 1.13 / 0.96, 5120 x 8192 1.13 / 0.96), 5 with two each below 4608 (4608 x 4096 1.12 / 0.98, 5120 x 4096 1.09 /
//     1.00), one a wave between (5120 x 5120 1.12 / 1.00);
//   11 or 12: 12 from 5120 on (6144 x 5120 1.00 / 0.95, x 12288 1.04 / 0.96, gated 1.05 / 0.96, fp8 1.01 / 0.93), 6 with two each below (6144 x 4096 0.97 / 0.95);
//   17 .. 20: 10 with two each in bf16, and in 8 bits from 8192 on (9216 x 4096 1.01 / 0.94, x 12288 1.08 / 0.99, fp8 1.02 / 0.96; but fp8 10240 x 4096 0.90 / 0.94);
//   hundreds (vocabularies in 8 bits): 12 (152064 x 5120 fp8 122.4 / 117.7 us).
// Over 870 shapes of 3072 to 27648 rows and K 2560 to 12288 in the three formats, the calls that come here take 0.935 of gemv_ldsx_kernel's time in the mean.  What still loses, 1 .. 3 %: 14336
// and 18432 rows with K of 8192 and more, 27648 x 12288 gated in bf16.  Four rows a task instead of two: the same within 2 %.
static int ring_waves(const ChattsLinearArgs* a) {
  const int cus = device_cus(), tasks = a->n / 2, each = (tasks + cus - 1) / cus;
  if (tasks / cus >= 128) return 12;
  if (each >= 5 && each <= 8) return tasks % cus == 0 ? each : 8;
  if (each == 9 || each == 10) return a->k >= 8192 ? 12 : (a->k < 4608 ? 5 : each);
  if (each == 11 || each == 12) return a->k >= 5120 ? 12 : 6;
  if (each >= 17 && each <= 20 && (!a->w8 || a->k >= 8192)) return 10;
  return 8;
}
// Measured in a graph over rotating weights, gemv_ldsx_kernel / here, us: bf16 24576 x 4096 gated 34.3 / 31.4, 4096 x 12288 19.8 / 18.2, 6144 x 4096 10.8 / 10.2, 4096 x 4096 8.2 / 7.8,
// 7168 x 5120 14.9 / 13.0, 5120 x 13824 25.4 / 24.4, 12288 x 3072 14.7 / 13.9; fp8 24576 x 4096 gated 21.1 / 17.4, 27648 x 5120 gated 26.7 / 23.5, 4096 x 12288 12.2 / 11.4, 7168 x 5120
// 9.7 / 8.3, 152064 x 5120 127 / 122; int8 24576 x 4096 gated 22.0 / 19.0, 4096 x 12288 12.5 / 11.2.
int launch_gemv_ring(const GemvParams& from, const ChattsLinearArgs* a, hipStream_t s) {
  GemvParams p = from;
  const int cus = device_cus();
  int nw = opt_get(OPT_GEMV_NW, ring_waves(a));
  if (nw < 1 || nw > 16) nw = 8;
  p.tasks = a->n / 2;                                     // two rows, gated: a gate and its up row
  p.spread = gemv_spread(a->w8 ? (size_t)a->ldw8 : (size_t)a->ldw * 2, (a->k + (a->w8 ? 1023 : 511)) / (a->w8 ? 1024 : 512));
  int grid = (p.tasks + nw - 1) / nw;
  const int most = cus * (opt_get(OPT_GEMV_OCC, 1) > 0 ? opt_get(OPT_GEMV_OCC, 1) : 1);
  if (grid > most) grid = most;
  const dim3 blocks(grid, a->batch > 1 ? a->batch : 1);
  const size_t lds = ring_lds(a);
  const bool norm = a->norm_w != nullptr;
  if (!a->w8) launch_ring_e<kFmtBf16>(p, a->epilogue, norm, blocks, nw * 64, lds, s);
  else if (a->w8_format == CHATTS_W8_INT8) launch_ring_e<CHATTS_W8_INT8>(p, a->epilogue, norm, blocks, nw * 64, lds, s);
  else launch_ring_e<CHATTS_W8_FP8>(p, a->epilogue, norm, blocks, nw * 64, lds, s);
  CHATTS_CHECK_LAUNCH("gemv_ring");
  return CHATTS_OK;
}

}  // namespace chatts
