// gemv4.h - what the two kernels of one row on 4-bit codes share (gemv4.hip: codes as a checkpoint holds them, gemv4_tiles.hip: codes laid out once)
#pragma once
#include "common.h"
#include "gemv_common.h"

namespace chatts {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

struct Gemv4Params {
  const uint8_t* w4;
  const float2* sz;
  const float* x;
  const float* norm_w;
  const float* bias;
  const float* resid;
  float* out;
  float eps;
  int n, k, ldw4, gshift, ng;
  int quads_each, quads_more;      // every workgroup has quads_each quads, the first quads_more of them one more
  unsigned parts_inv;              // ceil(2^32 / parts of K), 0 where there is one: a quotient without a division
};

constexpr int kQ4Waves = 8, kQ4Threads = 64 * kQ4Waves, kQ4Turns = 4;
constexpr int kQ4Piece = 512 + 32;      // bytes of an operand: (k group) x (part, hi / lo) x 16; the 32 keep the writes of x apart
constexpr unsigned kQ4Far = 0x7ffffff0u;
__host__ __device__ constexpr int q4_parts(int k) { return (k + 511) >> 9; }
static inline size_t q4_lds(int k, int quads, int waves) { return (size_t)q4_parts(k) * 4 * kQ4Piece + (size_t)quads * waves * 128; }

// quad q of a workgroup: its first row (gated: gates 2 u, 2 u + 1 and their up rows, 16 further on)
template <bool GLU>
__device__ __forceinline__ int q4_first_row(int q) {
  const int at = q * (GLU ? 2 : 4);
  return GLU ? (at >> 4) * 32 + (at & 15) : at;
}
// part [quad][wave][8] -> out: the quads of a workgroup x the units of K were dealt evenly over the waves, `items` of them, S a quad
template <int EPI, bool NORM, int WAVES>
__device__ __forceinline__ void q4_finish(const Gemv4Params& p, const f32x4* part, const float* red, int tid, int q0, int nq, int S, int items) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr bool GLU = epi_is_glu(EPI);
  const int K = p.k;
  float rstd = 1.f;
  if (NORM) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) t += red[i];
    rstd = rsqrtf(t / (float)K + p.eps);
  }
  // eight lanes a quad: the vectors of the waves that had a share of it, in wave order, then over the lanes
  for (int i = tid; i < (nq * 8 + 63) / 64 * 64; i += WAVES * 64) {
    const int qq = i >> 3, e = i & 7;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (qq < nq) {
      const int a = qq * S, z = a + S;
      // from the wave before the one that a 1 / items in floating point names: its share may end at a
      int w = (int)((float)(a * WAVES) * __builtin_amdgcn_rcpf((float)items)) - 1;
      for (w = w < 0 ? 0 : w; w < WAVES && w * items / WAVES < z; ++w) {
        const int to = (w + 1) * items / WAVES;
        if (to > a && w * items / WAVES < to) v += part[(qq * WAVES + w) * 8 + e];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] += lane_xor1(v[j]); v[j] += lane_xor2(v[j]); v[j] += half_mirror(v[j]); if (NORM) v[j] *= rstd; }
    if (qq >= nq) continue;
    const int row = q4_first_row<GLU>(q0 + qq);
    if (GLU) {
      if (e < 2) {
        float g = e ? v[2] : v[0], u = e ? v[3] : v[1];
        if (p.bias) { g += p.bias[row + e]; u += p.bias[row + e + 16]; }
        p.out[(q0 + qq) * 2 + e] = silu_f(g) * u;
      }
    } else if (e < 4) {
      float o = e == 0 ? v[0] : (e == 1 ? v[1] : (e == 2 ? v[2] : v[3]));
      if (p.bias) o += p.bias[row + e];
      if (EPI == CHATTS_EPI_RESID) o = p.resid[row + e] + o;
      p.out[row + e] = o;
    }
  }
#endif
}

}  // namespace chatts
