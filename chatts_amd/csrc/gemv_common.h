// gemv_common.h - the arithmetic of the batch-1 weight-streaming GEMV, shared by gemv.hip and gemv_ring.hip so that both
// accumulate a row in exactly the same order (bit-identical results).
#pragma once
#include "common.h"
#include "tp_common.h"

namespace chatts {

__device__ __forceinline__ float dot8(const u32x4 wv, const f32x4 xa, const f32x4 xb, float acc) {
  acc = fmaf(bf16_lo(wv.x), xa.x, acc);
  acc = fmaf(bf16_hi(wv.x), xa.y, acc);
  acc = fmaf(bf16_lo(wv.y), xa.z, acc);
  acc = fmaf(bf16_hi(wv.y), xa.w, acc);
  acc = fmaf(bf16_lo(wv.z), xb.x, acc);
  acc = fmaf(bf16_hi(wv.z), xb.y, acc);
  acc = fmaf(bf16_lo(wv.w), xb.z, acc);
  acc = fmaf(bf16_hi(wv.w), xb.w, acc);
  return acc;
}

// one RMSNorm partial-sum step (Qwen2RMSNorm: sum of squares in float32); ONE definition = one contraction pattern everywhere
__device__ __forceinline__ float sumsq4(float ss, const f32x4 v) {
  ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
  return ss;
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }

template <int ROWS, int EPI>
__device__ __forceinline__ int task_row(int task, int r) {
  if (epi_is_glu(EPI)) {   // gate/up interleaved in blocks of 16 rows: unit u -> rows g(u), g(u)+16
    const int unit = task * (ROWS / 2) + (r >> 1);
    return (unit >> 4) * 32 + (unit & 15) + (r & 1) * 16;
  }
  return task * ROWS + r;
}


struct GemvParams {
  const uint16_t* w;
  const float* x;
  const float* bias;
  const float* resid;
  float* out;
  const float* norm_w;
  float eps;
  int n;       // weight rows
  int k;
  int ldw;
  int tasks;   // number of row-group tasks
  const uint8_t* w8;      // fp8 (OCP e4m3fn) weights [N, ldw8] or NULL
  const float* w8_scale;  // per-row power-of-two scale: w = scale[row] * float(w8)
  int ldw8;
  int w8_format;          // CHATTS_W8_FP8 / CHATTS_W8_INT8
  // optional 4-bit copy of W (GPTQ codes, row-major: byte j of a row = codes 2j | 2j+1 << 4) with one (scale, scale * zero) pair
  // per `w4_group` weights of a row: w = bf16_rne(q * scale - scale_zero) - exactly the bf16 matrix the other kernels stream
  const uint8_t* w4;
  const float* w4_sz;     // [N, K / w4_group, 2]
  int ldw4, w4_group;
  TpParams tp;            // kEpiResidTp only
  int spread;             // chunks of K that a task may start with (gemv_first_chunk), 0: the first
  int ks;                 // gemv_ksplit_kernel: waves per row group
  float glu_limit, glu_alpha;   // CHATTS_EPI_CLAMPGLU
  int64_t x_stride, w_stride, out_stride;   // grid y: further products of the same shape
};

// The chunk of K that a task starts with.  Rows a multiple of 4 KB apart begin on the same memory channels and banks, and waves that walk such rows in step meet there:
// 24576 x 4096 bf16 took 38.8 us (41.4 without pairs), 31.5 with every four rows starting at a hashed chunk (a quarter of the rows' number, without a hash: 33.7 - the channels
// are themselves sums of address bits); 151936 x 4096 184.8 -> 177.3, 6144 x 4096 10.5 -> 10.0, 4096 x 4096 8.5 -> 8.1.  Other strides (5120, 13824 columns: 1 % slower) keep
// their order.  The row decides, not the geometry: ROWS, UNR and the exchange over ranks sum in the same order.
template <int ROWS>
__device__ __forceinline__ int gemv_first_chunk(int task, int spread) {
  return __builtin_amdgcn_readfirstlane((int)__umulhi((unsigned)(task * ROWS / 4) * 0x9E3779B1u, (unsigned)spread));
}
template <int EPI>
__device__ __forceinline__ float gemv_gated(const GemvParams& p, int rg, float g, float v) {
  if (p.bias) { g += p.bias[rg]; v += p.bias[rg + 16]; }
  return EPI == CHATTS_EPI_CLAMPGLU ? clamp_glu(g, v, p.glu_limit, p.glu_alpha) : (EPI == CHATTS_EPI_GEGLU ? gelu_tanh_glu(g, v) : silu_f(g) * v);
}
template <int EPI>
__device__ __forceinline__ float gemv_value(const GemvParams& p, int row, float v) {
  if (p.bias) v += p.bias[row];
  if (EPI == CHATTS_EPI_RESID) v = p.resid[row] + v;
  if (EPI == CHATTS_EPI_RELU2) { v = fmaxf(v, 0.f); v *= v; }
  return v;
}
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot16_fp8(const u32x4 wv, const f32x4 x0, const f32x4 x1, const f32x4 x2, const f32x4 x3,
                                            float acc) {
  f32x2 a;
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.x, false); acc = fmaf(a.x, x0.x, acc); acc = fmaf(a.y, x0.y, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.x, true);  acc = fmaf(a.x, x0.z, acc); acc = fmaf(a.y, x0.w, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.y, false); acc = fmaf(a.x, x1.x, acc); acc = fmaf(a.y, x1.y, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.y, true);  acc = fmaf(a.x, x1.z, acc); acc = fmaf(a.y, x1.w, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.z, false); acc = fmaf(a.x, x2.x, acc); acc = fmaf(a.y, x2.y, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.z, true);  acc = fmaf(a.x, x2.z, acc); acc = fmaf(a.y, x2.w, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.w, false); acc = fmaf(a.x, x3.x, acc); acc = fmaf(a.y, x3.y, acc);
  a = __builtin_amdgcn_cvt_pk_f32_fp8(wv.w, true);  acc = fmaf(a.x, x3.z, acc); acc = fmaf(a.y, x3.w, acc);
  return acc;
}

// int8 form of the same 16 weights: four sign-extended bytes per dword (v_cvt_f32_i32 with an SDWA byte select, or a bit-field extract
// before it - the compiler's choice), the same float32 FMAs.  |q| <= 127: the products are exact as in the fp8 form.
__device__ __forceinline__ float dot16_i8(const u32x4 wv, const f32x4 x0, const f32x4 x1, const f32x4 x2, const f32x4 x3, float acc) {
  auto four = [&](uint32_t d, const f32x4 x) {
    acc = fmaf((float)(int)(int8_t)(d & 0xffu), x.x, acc);
    acc = fmaf((float)(int)(int8_t)((d >> 8) & 0xffu), x.y, acc);
    acc = fmaf((float)(int)(int8_t)((d >> 16) & 0xffu), x.z, acc);
    acc = fmaf((float)((int)d >> 24), x.w, acc);
  };
  four(wv.x, x0); four(wv.y, x1); four(wv.z, x2); four(wv.w, x3);
  return acc;
}


// host: chunks of K that a task may start with
inline int gemv_spread(size_t row_bytes, int nchunks) { return row_bytes % 4096 == 0 ? nchunks : 0; }
// host: default waves per workgroup / workgroups per CU of the stand-alone bf16 GEMV (gemv.hip)
void gemv_default_geometry(int n, int k, int epilogue, int cus, int* nw_out, int* occ_out);

}  // namespace chatts
