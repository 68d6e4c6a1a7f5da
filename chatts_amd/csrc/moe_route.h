// moe_route.h - the choice of experts for a row by one wave (moe.hip; depth.hip, where the norm before the router chooses, too)
#pragma once
#include "common.h"

namespace chatts {

// what is chosen for a row: lane j has choice j
struct MoeChoice {
  int own, id;              // output, expert (-1: an identity output, or none)
  float mine;               // its score or logit
  float total, kept;        // sums over the choices: scores, those of identity outputs
};
__device__ __forceinline__ int moe_route_end(const ChattsMoeArgs& p, int row, int lane, bool parked, MoeChoice c) {
  if (p.choose == CHATTS_CHOOSE_LOGITS) {      // softmax over the chosen logits
    const float mx = wave_max(c.mine);
    c.mine = lane < p.top ? expf(c.mine - mx) : 0.f;
    c.total = wave_sum(c.mine);
    c.kept = wave_sum(c.own >= p.experts ? c.mine : 0.f);
  }
  const float inv = p.choose == CHATTS_CHOOSE_SCORES ? p.weight_scale : 1.0f / (c.total + 1e-20f);
  const int id = parked ? -1 : c.id;
  if (lane < p.top) {
    p.ids[(size_t)row * p.top + lane] = id;
    p.weight[(size_t)row * p.top + lane] = c.mine * inv;
    p.place[(size_t)row * p.top + lane] = -1;
  }
  if (lane == 0) p.kept[row] = parked ? 0.f : c.kept * inv;
  return id;
}

// Up to 64 outputs without choice groups: a lane an output (z: its logit), nothing goes through LDS.  Returns the expert of choice `lane`.
__device__ __forceinline__ int moe_route_row64(const ChattsMoeArgs& p, int row, int lane, float z) {
  const int N = p.experts + p.identity;
  const bool in = lane < N, logits = p.choose == CHATTS_CHOOSE_LOGITS;
  const int at = in ? lane : 0;
  const float cor = p.correction ? p.correction[at] : 0.f;
  const bool parked = p.rows[row].pos < 0;
  float sc = z;
  if (!logits) {
    const float mx = wave_max(in ? z : -INFINITY);
    const float e = in ? expf(z - mx) : 0.f;
    sc = e / wave_sum(e);
  }
  const float c0 = sc + cor;
  float ch = in && c0 > -INFINITY ? c0 : -INFINITY;      // (NaN is never chosen)
  MoeChoice c{-1, -1, logits ? -INFINITY : 0.f, 0.f, 0.f};
  for (int j = 0; j < p.top; ++j) {
    const float m = wave_max(ch);
    if (m == -INFINITY) break;                           // (nothing left)
    const int b = (int)__builtin_ctzll(__ballot(ch == m));
    const float s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc), b));
    if (lane == b) ch = -INFINITY;
    c.total += s;
    if (b >= p.experts) c.kept += s;
    if (lane == j) { c.own = b; c.id = b < p.experts ? b : -1; c.mine = s; }
  }
  return moe_route_end(p, row, lane, parked, c);
}

}  // namespace chatts
