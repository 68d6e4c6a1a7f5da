// gemm_ring.hip - the prefill projection (M > 16 rows on pre-split bf16 hi / lo planes of A):  C = epilogue(A . W^T), bf16x2.
// Round 5 rebuild of the LDS-DMA kernel (gemm_dma_kernel, round 1-4).  What the round-5 timeline probe of that kernel showed
// (tools/gemm_probe.py, profiles/r5_gemm_probe_before.txt) and what this kernel does about it:
//
//  1. The K loop was LOADER-bound, not MFMA-bound.  With two 64 KB stages a stage can only be requested after the barrier that
//     retires its slot and must have landed by the next barrier: 16 pieces per loader wave at ~100 cycles of issue each, then the
//     drain (vmcnt(0)), once per K-step - 2400-2500 cycles per step whatever the clock, against 2048 cycles of MFMA (a ragged tile
//     with a quarter of the MFMAs still took 1500).  HERE: the ring holds FOUR half-stages (32 K-values each, rows of 64 bytes); a
//     half-stage is requested three half-steps before it is needed, the loaders wait with a COUNTED vmcnt (two younger half-stages
//     stay in flight across every barrier) and never drain.  One barrier per half-step, placed between the lo and the hi sweep.
//  2. Every workgroup paid dispatch + prologue (~4.5 us per tile) and the epilogues ran as chains of dependent memory round trips
//     (direct stores 14 us, residual epilogue 25 us per tile: one `s_waitcnt vmcnt(0)` per element).  HERE: 256 PERSISTENT
//     workgroups walk their units; the loader waves run ahead into the next unit while the compute waves store; the MFMA operands
//     are swapped (D = W . A^T), so a lane holds 4 consecutive output columns of one token and the epilogue is branch-free 16-byte
//     loads / stores selected once per unit.
//  3. Tiles did not fill rounds of workgroups: 798 rows = 6 tiles of 128 + a ragged one of 30 (its second wave row idle, DMA-bound);
//     o_proj / down_proj ran 420 units (split-K 3) as two rounds on 256 CUs with a third of the CU-time idle.  HERE: the 16-row
//     fragments of M are dealt EVENLY over T M-tiles (50 fragments: 9,9,8,8,8,8 or 8,7,7,7,7,7,7 or 6,6,6,6,6,5,5,5,5), a tile's
//     fragments evenly over the two wave rows, and (T, split-K) are chosen per shape so that the units fill whole rounds
//     (o / down: 6 x 20 x 2 = 240 units; qkv: 9 x 28 = 252; gate_up: 7 x 108 = 756 = 2.95 rounds).
//
// Geometry: unit = (K split, W panel of 256 rows (or 192: NF), M-tile of f <= 10 fragments); 12 waves = 8 compute (2 x 4: wave row r holds
// ceil / floor of f / 2 fragments x 64 columns) + 4 loaders.  Half-stage slot (36 KB): A_hi [160][64 B] | A_lo | W [256][64 B]; 16-byte
// chunk c of row r lives at chunk c ^ (((r >> 3) & 1) << 1) (conflict-free for the ds_read_b128 fragment reads; applied on the SOURCE
// side of the DMA: lane l of a 16-row piece fetches global chunk (l & 3) ^ ((l >> 5) << 1)).
// Same products and the same per-element summation order over K as the kernels in gemm.hip at equal split-K.
#include <type_traits>

#include "gemm_common.h"
#include "ring_store.h"

namespace chatts {

constexpr int kRingBN = kRingPanel, kRingMaxF = 10, kRingSlots = 4;
constexpr int kRingAPlane = kRingMaxF * 16 * 64;             // 10 KB: one plane of a half-stage
constexpr int kRingWOff = 2 * kRingAPlane;
constexpr int kRingHalf = kRingWOff + kRingBN * 64;          // 36 KB
constexpr int kRingLds = kRingSlots * kRingHalf;             // 144 KB
constexpr int kRingThreads = 768, kRingCompute = 8, kRingLoaders = 4;


// GROUPED (launch_ring_group): unit = (W panel, tile of a list), the tiles' number is only known on the device.  All panels of two tiles (an expert's, mostly) come one after the other: the
// panels on an XCD then read the same rows of A at the same time, which are 1.2 GB of half lines a layer out of L2 or from behind it, and those of 16 experts do not fit beside the weights
// that stream.  us for both products of 32 experts, 4 a token, 4096 x 1536, panel by panel over all tiles / so: 400 tokens 303 / 290, 700 353 / 330, 1024 420 / 392, 2048 650 / 608; one
// tile instead of two 289, 333, 395, 618, four 298, 338, 402, 613.
constexpr int kRingGroupTiles = 2;
__device__ __forceinline__ RingUnit ring_group_unit(const GemmParams& p, const RingGroup& gr, int T, int P, int u, int& matrix, int& places) {
  RingUnit r;
  const int first = u / (kRingGroupTiles * P) * kRingGroupTiles, at = u - first * P, n = T - first < kRingGroupTiles ? T - first : kRingGroupTiles;
  const int32_t* t = gr.tiles + (size_t)(first + at % n) * 4;
  matrix = t[0];
  r.m0 = t[1];
  places = t[2];
  r.panel = at / n;
  r.split = 0;
  r.f = (places + 15) >> 4;
  r.f0 = (r.f + 1) >> 1;
  r.kbeg = 0;
  r.nh = p.k >> 5;
  return r;
}

// Loader wave L over lists of rows: how many pieces a tile has is only known on the device, so a piece is a branch and a wait a choice at run time.  Planes row-major, four column fragments.
constexpr int kGroupNF = 4;
__device__ __forceinline__ void ring_group_load(const GemmParams& p, const RingGroup& gr, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, int T, int P, int u0, int uend, int ustep, int L,
                                                int lane, char* smem) {
  const int prow = lane >> 2, gchunk = (lane & 3) ^ ((lane >> 5) << 1);
  const bool wtiled = p.wt != nullptr;
  const int nkt = p.k >> 5, wstep = wtiled ? 1024 : 64;
  const char* src[kGroupNF + 5];
  int dst[kGroupNF + 5];
  int np = 0, hh = 0, ucur = u0;
  auto setup = [&](int u) {
    int matrix = 0, places = 0;
    const RingUnit r = ring_group_unit(p, gr, T, P, u, matrix, places);
    const int n0 = r.panel * kRingBN;
    const size_t skip = (size_t)matrix * gr.w_stride;
#pragma unroll
    for (int h = 0; h < kGroupNF; ++h) {
      int wr = n0 + (L + 4 * h) * 16 + prow;
      if (wr > p.n - 1) wr = p.n - 1;
      if (wtiled) {
        const int rr = wr & 15;
        src[h] = reinterpret_cast<const char*>(p.wt + skip + (size_t)(wr >> 4) * nkt * 512) + (rr * 4 + (gchunk ^ ((rr >> 3) << 1))) * 16;
      } else {
        src[h] = reinterpret_cast<const char*>(p.w + skip + (size_t)wr * p.ldw + gchunk * 8);
      }
      dst[h] = kRingWOff + (L + 4 * h) * 1024;
    }
    np = kGroupNF;
#pragma unroll
    for (int h = 0; h < 5; ++h) {
      const int q = L + 4 * h;
      if (q < 2 * r.f) {
        const int plane = q >= r.f, frag = plane ? q - r.f : q;
        int am = r.m0 + frag * 16 + prow;
        if (am > r.m0 + places - 1) am = r.m0 + places - 1;
        if (gr.order) am = gr.order[am] / gr.top;
        src[kGroupNF + h] = reinterpret_cast<const char*>((plane ? a_lo : a_hi) + (size_t)am * ldp + gchunk * 8);
        dst[kGroupNF + h] = plane * kRingAPlane + frag * 1024;
        np = kGroupNF + 1 + h;
      }
    }
  };
  int gi = 0;                                                // global index of the next half-stage to request
  auto issue = [&]() -> int {                                // request the next half-stage (if any); -> its piece count
    if (ucur >= uend) return 0;
    char* base = smem + (gi & (kRingSlots - 1)) * kRingHalf;
    const size_t koffw = (size_t)hh * wstep, koffa = (size_t)hh * 64;
#pragma unroll
    for (int h = 0; h < kGroupNF + 5; ++h)
      if (h < np) __builtin_amdgcn_global_load_lds((gptr_t)(src[h] + (h < kGroupNF ? koffw : koffa)), (lptr_t)(base + dst[h]), 16, 0, 0);
    const int n = np;
    ++gi;
    if (++hh == nkt) {
      ucur += ustep;
      hh = 0;
      if (ucur < uend) setup(ucur);
    }
    return n;
  };
  const int G = (uend - u0 + ustep - 1) / ustep * nkt;       // half-steps of this workgroup = barriers after the first
  setup(u0);
  issue();
  int q1 = issue(), q2 = issue();
  ring_wait_vmcnt(q1 + q2);                                  // half-stage 0 landed
  __builtin_amdgcn_s_barrier();                              // ... published
  int q3 = issue();                                          // (slot 3 has never been read)
  for (int gh = 0; gh < G; ++gh) {
    ring_wait_vmcnt(q2 + q3);                                // half-stage gh + 1 landed; gh + 2, gh + 3 stay in flight
    __builtin_amdgcn_s_barrier();                            // publishes it; every read of half-stage gh has returned
    const int q4 = issue();                                  // gh + 4 -> the slot of gh
    q1 = q2; q2 = q3; q3 = q4;
  }
  (void)q1;
}

// SINGLE: the "bf16" speed mode - the lo plane is neither staged nor multiplied (activations rounded to bf16: NOT parity grade)
// NF: column fragments of a compute wave - a panel is 64 NF rows of W
// TILES: planes of A or of the result whose whole blocks lie in tiles and whose last rows do not (a_tiled, c_tiled).  An instance of its own: the choice a piece cost row-major planes up
// to 4 % (us with it / without, W in tiles: 300 rows 4096 x 4096 35.5 / 34.2, 12288 x 4096 gated 70.3 / 69.4; 700 rows 6144 x 4096 77.3 / 76.0; 129 rows 5120 x 5120 33.4 / 32.6; 2048 rows
// 12288 x 4096 gated 313.6 / 312.3).
template <bool SINGLE, bool GROUPED = false, int NF = 4, bool TILES = false>
__global__ __launch_bounds__(kRingThreads) void gemm_ring_kernel(GemmParams p, const uint16_t* __restrict__ a_hi,
                                                                 const uint16_t* __restrict__ a_lo, int ldp, RingGeom g, RingGroup gr) {
  static_assert(!GROUPED || (!SINGLE && NF == 4 && !TILES), "what the loader of lists knows");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BN = 64 * NF;
  kernarg_touch<sizeof(GemmParams) + 2 * sizeof(void*) + 8 + sizeof(RingGeom) + (GROUPED ? sizeof(RingGroup) : 0)>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this workgroup's units: XCD x (= blockIdx % 8, observed; speed only) owns a contiguous eighth of the unit sequence and its
  // workgroups take every wpx-th unit of it, so that at any time an XCD works on ~wpx consecutive units: the M-tiles of a few W panels
  // at the same K offset - each K-slice of a panel is fetched into that L2 once for all of them
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  if constexpr (GROUPED) {
    g.T = *gr.count;
    g.units = g.T * g.P;
  }
  auto unit = [&](int u, int& matrix, int& places) __attribute__((always_inline)) {
    if constexpr (GROUPED) return ring_group_unit(p, gr, g.T, g.P, u, matrix, places);
    else return ring_unit(p, g, u);
  };
  const int share = g.units >> 3, rem = g.units & 7;
  const int ubeg = xcd * share + (xcd < rem ? xcd : rem), ucnt = share + (xcd < rem);
  if (local >= ucnt) return;                                   // padding workgroup (fewer units than workgroups): uniform exit
  const int uend = ubeg + ucnt, u0 = ubeg + local, ustep = g.wpx;

  if (wave >= kRingCompute) {
    // ---- loader wave L: pieces of 16 rows x 64 bytes (1 KB per wave instruction).  W pieces {L, L + 4, L + 8, L + 12}; of the unit's
    // A pieces q = 0 .. 2 f - 1 (q < f: hi plane fragment q, else lo plane fragment q - f) those with q % 4 == L.
    const int L = wave - kRingCompute;
    if constexpr (GROUPED) {
      ring_group_load(p, gr, a_hi, a_lo, ldp, g.T, g.P, u0, uend, ustep, L, lane, smem);
    } else {
      const int prow = lane >> 2, gchunk = (lane & 3) ^ ((lane >> 5) << 1);
      // tiled operands (chatts_tile_bf16): piece (16-row block b, half-stage t) is the 1 KB at ((b * K / 32) + t) * 1 KB, already in LDS
      // order - whole cache lines per request instead of 16 half lines (profiles/r6_feed_probe.txt)
      const bool wtiled = p.wt != nullptr, alltiled = p.planes_tiled != 0;
      const int nkt = p.k >> 5, wstep = wtiled ? 1024 : 64, astep = alltiled ? 1024 : 64;
      // three fragments do not hold whole (gate, up) pairs of 16 columns: there a gated product's W block is 8 gates and their 8 up rows
      const bool mixed = NF == 3 && p.direct && epi_is_glu(p.epilogue);
      // A launch's first bytes wait for what stands here: places by multiplication, bases in scalar registers, one offset a lane (as divisions and 64-bit addresses a lane they took 1.4 to
      // 2.0 us of a launch).  As many pieces a half-stage for the whole launch (a shorter tile asks for one of its pieces twice): one loop, straight down, whose waits are constants (a branch
      // a piece and the choice of the wait at run time: 1 us).
      const int fmax = g.fbase + (g.frem > 0), na_max = SINGLE ? fmax : 2 * fmax, more = na_max > L ? (na_max - L + 3) >> 2 : 0;
      const int wl = mixed ? (L & 1) * 8 + (prow & 7) : prow;      // this lane's row of a tiled block of W
      unsigned lane_w = wtiled ? (mixed ? (unsigned)(prow >> 3) * (unsigned)nkt * 1024u : 0u) + (wl * 4 + (gchunk ^ ((wl >> 3) << 1))) * 16
                                     : (unsigned)(mixed ? (prow >> 3) * 16 + (prow & 7) : prow) * (unsigned)p.ldw * 2u + gchunk * 16;
      auto run = [&](auto n_c) __attribute__((always_inline)) {
        constexpr int N = decltype(n_c)::value, NA = N - NF;
        const char* wb[NF];
        const char* ab[NA > 0 ? NA : 1];
        unsigned lane_a[NA > 0 ? NA : 1];
        int to[NA > 0 ? NA : 1], ashift[NA > 0 ? NA : 1];
        char* base = smem;
        int left = 3;                                          // half-stages that are asked for before the first barrier
        for (int u = u0; u < uend; u += ustep) {
          const RingUnit r = ring_unit(p, g, u);
          const int kb = r.kbeg >> 5, na = SINGLE ? r.f : 2 * r.f;
#pragma unroll
          for (int h = 0; h < NF; ++h) {                       // (n is a multiple of 16, of 32 where it is gated: a block is there or not)
            if (mixed) {
              int unit8 = r.panel * (BN / 16) + L + 4 * h;     // eights of units
              if (unit8 > (p.n >> 4) - 1) unit8 -= ((unit8 - ((p.n >> 4) - 1) + 1) >> 1) << 1;      // (its parity is in lane_w)
              wb[h] = wtiled ? reinterpret_cast<const char*>(p.wt) + ((size_t)(unit8 >> 1) * 2 * nkt + kb) * 1024
                             : reinterpret_cast<const char*>(p.w) + ((size_t)((unit8 >> 1) * 32 + (unit8 & 1) * 8) * p.ldw + r.kbeg) * 2;
            } else {
              int rb = r.panel * (BN / 16) + L + 4 * h;
              if (rb > (p.n >> 4) - 1) rb = (p.n >> 4) - 1;
              wb[h] = wtiled ? reinterpret_cast<const char*>(p.wt) + ((size_t)rb * nkt + kb) * 1024 : reinterpret_cast<const char*>(p.w) + ((size_t)rb * 16 * p.ldw + r.kbeg) * 2;
            }
          }
#pragma unroll
          for (int h = 0; h < NA; ++h) {
            int q = L + 4 * h;
            if (q >= na) q = h > 0 ? q - 4 : na - 1;             // (two fewer than the most)
            const int plane = q >= r.f, frag = plane ? q - r.f : q, row = r.m0 + frag * 16;
            const bool atiled = TILES ? alltiled || row < p.a_tiled : alltiled;
            ashift[h] = atiled ? 10 : 6;
            to[h] = plane * kRingAPlane + frag * 1024;
            const char* pl = reinterpret_cast<const char*>(plane ? a_lo : a_hi);
            if (atiled) {
              ab[h] = pl + ((size_t)(row >> 4) * nkt + kb) * 1024;
              lane_a[h] = lane * 16;
            } else {
              ab[h] = pl + ((size_t)row * ldp + r.kbeg) * 2;
              const int last = p.m - 1 - row;
              lane_a[h] = (unsigned)(prow < last ? prow : last) * (unsigned)ldp * 2u + gchunk * 16;
            }
          }
          for (int t = 0; t < r.nh; ++t) {
            if (left > 0) {
              --left;
            } else {
              ring_wait_vmcnt_c<2 * N>();                      // the half-stage before the two youngest has landed
              __builtin_amdgcn_s_barrier();                    // publishes it; every read of the slot that is asked for next has returned
            }
            asm("" : "+v"(lane_w));                            // (the sum of base and offset is not one to be carried along in vector registers)
#pragma unroll
            for (int h = 0; h < NA; ++h) asm("" : "+v"(lane_a[h]));
#pragma unroll
            for (int h = 0; h < NF; ++h) {
              __builtin_amdgcn_global_load_lds((gptr_t)(wb[h] + lane_w), (lptr_t)(base + kRingWOff + (L + 4 * h) * 1024), 16, 0, 0);
              wb[h] += wstep;
            }
#pragma unroll
            for (int h = 0; h < NA; ++h) {
              __builtin_amdgcn_global_load_lds((gptr_t)(ab[h] + lane_a[h]), (lptr_t)(base + to[h]), 16, 0, 0);
              ab[h] += TILES ? 1 << ashift[h] : astep;
            }
            base = base == smem + (kRingSlots - 1) * kRingHalf ? smem : base + kRingHalf;
          }
        }
        // (a launch has two half-steps at least)
        if (left > 0) ring_wait_vmcnt_c<N>();
        else ring_wait_vmcnt_c<2 * N>();
        __builtin_amdgcn_s_barrier();
        if (left == 0) {
          ring_wait_vmcnt_c<N>();
          __builtin_amdgcn_s_barrier();
        }
        ring_wait_vmcnt_c<0>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
      };
      switch (more) {
        case 0: run(std::integral_constant<int, NF>{}); break;
        case 1: run(std::integral_constant<int, NF + 1>{}); break;
        case 2: run(std::integral_constant<int, NF + 2>{}); break;
        case 3: run(std::integral_constant<int, NF + 3>{}); break;
        case 4: run(std::integral_constant<int, NF + 4>{}); break;
        default: run(std::integral_constant<int, NF + 5>{}); break;
      }
    }
    return;
  }

  // ---- compute wave (wm, wn): wave row wm holds f0 (wm = 0) or f - f0 fragments of the tile, 64 columns wn * 64 ..
  const int wm = wave >> 2, wn = wave & 3;
  const int lane_off = (lane & 15) * 64 + ((((lane >> 4) ^ (((lane >> 3) & 1) << 1))) << 4);      // byte offset of this lane's chunk in a 16-row block
  __builtin_amdgcn_s_barrier();                                // half-stage 0 published
  int gh = 0;
  for (int u = u0; u < uend; u += ustep) {
    int matrix = 0, places = 0;
    const RingUnit r = unit(u, matrix, places);
    if constexpr (GROUPED) p.m = r.m0 + places;
    const int fml = wm ? r.f - r.f0 : r.f0;
    const int rowblk = wm ? r.f0 : 0;                          // first fragment of this wave within the tile
    if (fml == 0) {
      for (int h = 0; h < r.nh; ++h) __builtin_amdgcn_s_barrier();
      gh += r.nh;
      continue;
    }
    f32x4 acc[5][NF];
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    auto k_loop = [&](auto fml_c) {
      constexpr int FML = decltype(fml_c)::value;
      bf16x8_t wf[NF], alo[FML], ahi[FML];
      const int a_off = rowblk * 1024 + lane_off, w_off = kRingWOff + wn * NF * 1024 + lane_off;
      auto slot = [&](int h) { return smem + ((gh + h) & (kRingSlots - 1)) * kRingHalf; };
      auto read_a = [&](const char* base, int plane, bf16x8_t (&dst)[FML]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FML; ++i) dst[i] = *reinterpret_cast<const bf16x8_t*>(base + plane * kRingAPlane + a_off + i * 1024);
      };
      auto column = [&](int j, const bf16x8_t (&af)[FML]) __attribute__((always_inline)) {      // D = W . A^T: operands swapped
#pragma unroll
        for (int i = 0; i < FML; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
      };
      // Half-step h (operands in registers).  Behind the barrier the fragments of h + 1 are asked for: lo, then a column of W behind its last product and into its registers, hi behind the
      // last column.  (Both sweeps row by row, W in two sets and all of it asked for at once with lo: 224 rows 4096 x 4096 26.7 / 26.0 us, 4096 x 12288 53.5 / 52.5, 800 rows
      // 27648 x 5120 gated 334.6 / 333.5, 2048 rows the same.)
      auto half = [&](int h, auto more_c) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!SINGLE) {
#pragma unroll
          for (int j = 0; j < NF; ++j) column(j, alo);
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // every fragment read of half-stage h has returned
        __builtin_amdgcn_s_barrier();                          // h + 1 is published; the loaders refill the slot of h
        const char* nb = slot(h + 1);
        if constexpr (MORE && !SINGLE) read_a(nb, 1, alo);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NF; ++j) {
          column(j, ahi);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (MORE) wf[j] = *reinterpret_cast<const bf16x8_t*>(nb + w_off + j * 1024);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MORE) read_a(nb, 0, ahi);
      };
      {
        const char* b0 = slot(0);
        if constexpr (!SINGLE) read_a(b0, 1, alo);
#pragma unroll
        for (int j = 0; j < NF; ++j) wf[j] = *reinterpret_cast<const bf16x8_t*>(b0 + w_off + j * 1024);
        read_a(b0, 0, ahi);
      }
      // (nh is even: K splits are multiples of 64; the last pair is peeled so that the loop body has no test)
      int h = 0;
      for (; h + 2 < r.nh; h += 2) {
        half(h, std::true_type{});
        half(h + 1, std::true_type{});
      }
      half(h, std::true_type{});
      half(h + 1, std::false_type{});
    };
    switch (fml) {
      case 1: k_loop(std::integral_constant<int, 1>{}); break;
      case 2: k_loop(std::integral_constant<int, 2>{}); break;
      case 3: k_loop(std::integral_constant<int, 3>{}); break;
      case 4: k_loop(std::integral_constant<int, 4>{}); break;
      default: k_loop(std::integral_constant<int, 5>{}); break;
    }
    gh += r.nh;

    const int tok0 = r.m0 + rowblk * 16, fb0 = r.panel * BN + wn * 16 * NF;
    const bool planes = p.c_hi != nullptr;
    if (!p.direct) ring_store<kStRaw, false, TILES>(p, acc, fml, tok0, fb0, lane, r.split);
    else if (p.epilogue == CHATTS_EPI_SWIGLU) {
      if (planes) ring_store<kStSwiglu, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStSwiglu, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else if (p.epilogue == CHATTS_EPI_RESID) {
      if (planes) ring_store<kStResid, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStResid, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else if (p.epilogue == CHATTS_EPI_GELU) {
      if (planes) ring_store<kStGelu, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStGelu, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else if (p.epilogue == CHATTS_EPI_CLAMPGLU) {
      if (planes) ring_store<kStClampGlu, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStClampGlu, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else if (p.epilogue == CHATTS_EPI_GEGLU) {
      if (planes) ring_store<kStGeglu, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStGeglu, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else if (p.epilogue == CHATTS_EPI_RELU2) {
      if (planes) ring_store<kStRelu2, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStRelu2, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    } else {
      if (planes) ring_store<kStNone, true, TILES>(p, acc, fml, tok0, fb0, lane, 0);
      else ring_store<kStNone, false, TILES>(p, acc, fml, tok0, fb0, lane, 0);
    }
  }
}

// ---- host side ------------------------------------------------------------------------------------------------------------------
// (T, sk, panel) per shape: a cost model in cycles of the slowest workgroup - its K-steps, a constant per unit, the split-K epilogue launch.  Fitted to what its pick costs against the best
// of 16000 measurements, planes and W in tiles: 13 projections (K 2048 .. 13824, N 2048 .. 27648; epilogues none, GELU, gated, residual with the norm behind it) at 40 .. 2048 rows.  A 64-deep
// step of a tile with f fragments takes 260 f + 1045 cycles in panels of 256 rows, 214 f + 965 in panels of 192 (the 4 f NF MFMAs per SIMD and the (32 f + 64 NF) x 128 bytes of LDS-DMA
// overlap only partly); of several units a workgroup meets the longest tile once and the mean one else; a unit costs 4900 of prologue and stores, a split 5 us of epilogue (7 from five slabs on,
// 16 from nine on, which the row-wise norm cannot hold in registers) and its slab traffic at ~4 to 5 TB/s, less where the slabs outgrow 64 MB.  Over these its pick is 1.0 % slower than the best
// triple in the mean (1.1 up to 144 rows, 0.4 above 900; at most 10: 7168 x 5120, 80 rows); the constants before, fitted to row-major planes, the longest tile for every unit: 2.0 (3.6, 0.8; 46).
// us before / now: 5120 x 13824, 80 rows 57.8 / 41.9; 6144 x 4096, 384 rows 49.1 / 44.0; 4096 x 4096 GELU, 1036 rows 74.4 / 68.0; 7168 x 5120, 600 rows 86.7 / 81.1; 27648 x 5120 gated, 2048
// rows (13 tiles / 14: six rounds both) 883 / 830.  What lies on the wrong side by more than 1 %: 24576 x 4096 gated, 600 rows 191.8 / 197.9.
// Panels of 192 rows are dearer per column, but fill CUs that panels of 256 leave without a unit: 24576 x 4096 gated, 223 rows: 96 panels x 2 tiles on 192 CUs 94.6 us, 128 x 2 on 256 CUs 80.0.
void ring_pick(int m, int n, int k, int cus, int force_t, int force_sk, int force_nf, RingGeom& g) {
  const int F = (m + 15) / 16, nk = k / 64;
  g.F = F;
  const int slots = cus >= 8 ? (cus / 8) * 8 : 8;
  double best = 1e30;
  const int tmin = (F + kRingMaxF - 1) / kRingMaxF;
  int bt = tmin, bs = 1, bf = 4;
  int tmax = (F + 2) / 3;                              // >= 3 fragments per tile
  if (tmax < tmin) tmax = tmin;
  for (int nf = 4; nf >= 3; --nf) {
    if (force_nf && nf != force_nf) continue;
    const int P = (n + 64 * nf - 1) / (64 * nf);
    const double frag = nf == 4 ? 260.0 : 214.0, tile = nf == 4 ? 1045.0 : 965.0;
    for (int T = tmin; T <= tmax; ++T) {
      const int fmax = (F + T - 1) / T;
      const double most = frag * fmax + tile, mean = frag * F / T + tile;
      // the work itself, evenly spread over the CUs: its fragments and a constant a tile, so more tiles only add to it
      if (mean * T * P * nk > best * slots) break;
      for (int sk = 1; sk <= 16; ++sk) {
        if (sk > 1 && nk / sk < 4) break;
        const long long units = (long long)T * P * sk;
        const long long rounds = (units + slots - 1) / slots;
        const int steps = (nk + sk - 1) / sk;
        double t = steps * (most + (double)(rounds - 1) * mean) + rounds * 4900.0;
        if (sk > 1) {
          const double slabs = (double)m * n * 4.0;
          t += (sk <= 4 ? 10300.0 : sk <= 8 ? 14200.0 : 34000.0) + (sk + 2) * slabs / (sk * slabs > 64e6 ? 1365.0 : sk <= 4 ? 2200.0 : 1770.0);
        }
        // a split that is no more than 0.7 % nearer counts as equal: slabs are the part that the model knows least
        if (sk > 1) t *= 1.007;
        if (t < best) { best = t; bt = T; bs = sk; bf = nf; }
      }
    }
  }
  if (force_t >= tmin && force_t <= F) bt = force_t;
  if (force_sk >= 1 && force_sk <= 16 && nk / force_sk >= 1) bs = force_sk;
  g.T = bt; g.sk = bs; g.nf = bf;
  g.P = (n + 64 * bf - 1) / (64 * bf);
  g.units = bt * g.P * bs;
  int wpx = (g.units + 7) / 8;
  if (wpx > slots / 8) wpx = slots / 8;
  g.wpx = wpx;
}

template <bool SINGLE, int NF, bool TILES>
static int launch_ring_n(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGeom& g, hipStream_t s) {
  static bool configured = false;     // > 64 KB of dynamic LDS must be opted into once
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<SINGLE, false, NF, TILES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             kRingLds);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemm_ring: cannot reserve %d bytes of LDS: %s", kRingLds, hipGetErrorString(e));
    configured = true;
  }
  hipLaunchKernelGGL((gemm_ring_kernel<SINGLE, false, NF, TILES>), dim3(8 * g.wpx), dim3(kRingThreads), kRingLds, s, p, a_hi, a_lo, ldp, g, RingGroup{});
  return CHATTS_OK;
}
template <bool SINGLE, int NF>
static int launch_ring_t(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGeom& g, hipStream_t s) {
  return p.a_tiled || p.c_tiled ? launch_ring_n<SINGLE, NF, true>(p, a_hi, a_lo, ldp, g, s) : launch_ring_n<SINGLE, NF, false>(p, a_hi, a_lo, ldp, g, s);
}
int launch_ring_group(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGroup& gr, int most_tiles, hipStream_t s) {
  static_assert(kRingTile == kRingMaxF * 16, "a tile's places");
  CHATTS_REQUIRE(!p.planes_tiled && !p.a_tiled && !p.c_tiled && p.direct && p.k % 64 == 0, CHATTS_E_SHAPE, "gemm_ring_group: row-major planes, K in one piece of whole steps (K=%d)", p.k);
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<false, true>), hipFuncAttributeMaxDynamicSharedMemorySize, kRingLds);
    CHATTS_REQUIRE(e == hipSuccess, CHATTS_E_LAUNCH, "gemm_ring: cannot reserve %d bytes of LDS: %s", kRingLds, hipGetErrorString(e));
    configured = true;
  }
  RingGeom g{};
  g.P = (p.n + kRingBN - 1) / kRingBN;
  const int cus = device_cus(), most = (most_tiles * g.P + 7) / 8;
  g.wpx = cus / 8 < most ? cus / 8 : most;
  if (g.wpx < 1) g.wpx = 1;
  hipLaunchKernelGGL((gemm_ring_kernel<false, true>), dim3(8 * g.wpx), dim3(kRingThreads), kRingLds, s, p, a_hi, a_lo, ldp, g, gr);
  CHATTS_CHECK_LAUNCH("gemm_ring_group");
  return CHATTS_OK;
}
int launch_ring(const GemmParams& p, const uint16_t* a_hi, const uint16_t* a_lo, int ldp, const RingGeom& geom, bool single, hipStream_t s) {
  RingGeom g = geom;
  g.finish();
  if (g.nf == 3) return single ? launch_ring_t<true, 3>(p, a_hi, a_lo, ldp, g, s) : launch_ring_t<false, 3>(p, a_hi, a_lo, ldp, g, s);
  return single ? launch_ring_t<true, 4>(p, a_hi, a_lo, ldp, g, s) : launch_ring_t<false, 4>(p, a_hi, a_lo, ldp, g, s);
}

// bf16 [rows, k] row-major -> the tiled layout: block (b = row / 16, t = k / 32) is 1 KB at ((b * k / 32) + t) * 1 KB; inside it the 16-byte
// chunk at position l (0 .. 63) holds row 16 b + (l >> 2), K-values 32 t + 8 c .. + 7 with c = (l & 3) ^ ((l >> 5) << 1) - the order in
// which the lanes of an LDS-DMA piece deposit a half-stage block (the header comment's swizzle).  Rows beyond the matrix repeat the last row.
__global__ __launch_bounds__(256) void tile_bf16_kernel(const uint16_t* __restrict__ src, int rows, int k, int ld, uint16_t* __restrict__ dst) {
  const int nkt = k >> 5;
  const size_t chunks = (size_t)((rows + 15) >> 4) * nkt * 64;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (size_t)gridDim.x * 256) {
    const int l = (int)(i & 63);
    const size_t blk = i >> 6;
    const int t = (int)(blk % nkt);
    int row = (int)(blk / nkt) * 16 + (l >> 2);
    if (row > rows - 1) row = rows - 1;
    const int c = (l & 3) ^ ((l >> 5) << 1);
    *reinterpret_cast<u32x4*>(dst + i * 8) = *reinterpret_cast<const u32x4*>(src + (size_t)row * ld + t * 32 + c * 8);
  }
}

}  // namespace chatts

extern "C" size_t chatts_tile_bf16_elems(int rows, int k) { return rows > 0 && k > 0 ? (size_t)((rows + 15) / 16) * 16 * k : 0; }

extern "C" int chatts_tile_bf16(const chatts_bf16* src, int rows, int k, int ld, chatts_bf16* dst, chatts_stream_t stream) {
  using namespace chatts;
  CHATTS_REQUIRE(rows >= 0 && k > 0 && k % 32 == 0 && ld >= k && ld % 8 == 0, CHATTS_E_SHAPE, "tile_bf16: rows=%d k=%d ld=%d (K %% 32 == 0, ld %% 8 == 0)", rows, k, ld);
  if (rows == 0) return CHATTS_OK;
  CHATTS_REQUIRE(src && dst && ((uintptr_t)src % 16) == 0 && ((uintptr_t)dst % 16) == 0, CHATTS_E_BADARG, "tile_bf16: null / unaligned pointer");
  const size_t chunks = chatts_tile_bf16_elems(rows, k) / 8;
  const unsigned blocks = (unsigned)((chunks + 255) / 256 < 16384 ? (chunks + 255) / 256 : 16384);
  hipLaunchKernelGGL(tile_bf16_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), src, rows, k, ld, dst);
  CHATTS_CHECK_LAUNCH("tile_bf16");
  return CHATTS_OK;
}

