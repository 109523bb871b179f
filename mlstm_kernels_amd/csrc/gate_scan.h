// Within-chunk scans of the gates by one wave, two positions per lane (gates.hip has the formulas): for the gate pre-pass and for the
// kernels that make their own gate vectors.
#pragma once
#include "common.h"

namespace mlstm {

// Scans over the 64 lanes by cross-lane moves of the vector unit where it has them: a shuffle through LDS takes ten times as long, and a
// chunk needs over twenty scan steps one after the other (8 heads of 317 positions of 256/512, short_fw with its own gates: 14.05 us by
// shuffles, 13.5 with the sums in another order).
__device__ __forceinline__ float lane_up(float x, float first) {  // of the lane before
  return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(first), __float_as_uint(x), 0x138, 0xf, 0xf, false));  // wave_shr:1
}
// Inclusive sums.  Step o adds the sum of the o lanes before to that of the last o: the order of the sums is that of six shuffles.
__device__ __forceinline__ float wave_incl_sum(float x) {
  float y = lane_up(x, 0.f);
  x = y + x;
  y = lane_up(lane_up(x, 0.f), 0.f);
  x = y + x;
  y = lane_up(lane_up(lane_up(lane_up(x, 0.f), 0.f), 0.f), 0.f);
  x = y + x;
#pragma unroll
  for (int o = 8; o < 64; o <<= 1) {
    y = __shfl_up(x, o);
    x = (int)(threadIdx.x & 63) >= o ? y + x : x;
  }
  return x;
}
__device__ __forceinline__ float wave_rev_incl_sum(float x) {  // over the lanes from this one on
  return __shfl_xor(wave_incl_sum(__shfl_xor(x, 63)), 63);
}
// Inclusive maxima (in any order the same): inside rows of 16 lanes, then row by row.
__device__ __forceinline__ float wave_incl_max(float x) {
#define MLSTM_DPP_MAX(ctrl, rows)                                                                                                  \
  x = fmaxf(__uint_as_float(__builtin_amdgcn_update_dpp(0xff800000u, __float_as_uint(x), ctrl, rows, 0xf, false)), x);
  MLSTM_DPP_MAX(0x111, 0xf)  // row_shr:1, 2, 4, 8
  MLSTM_DPP_MAX(0x112, 0xf)
  MLSTM_DPP_MAX(0x114, 0xf)
  MLSTM_DPP_MAX(0x118, 0xf)
  MLSTM_DPP_MAX(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
  MLSTM_DPP_MAX(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef MLSTM_DPP_MAX
  return x;
}
__device__ __forceinline__ float last_lane(float x) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 63)); }

// The gates of a lane's positions as they lie in memory: requested in one place, converted where they are used (positions past the
// end: the last one again, see scan_chunk).
struct RawGates {
  uint32_t i[2], f[2];
};
__device__ __forceinline__ RawGates load_gates(const void* ig, const void* fg, int bh, int c, int lane, int S, int dtype) {
  RawGates x;
  const int t0 = c * kChunk + 2 * lane;
  const size_t o0 = (size_t)bh * S + min(t0, S - 1), o1 = (size_t)bh * S + min(t0 + 1, S - 1);
  if (dtype == 0) {
    x.i[0] = ((const uint32_t*)ig)[o0], x.i[1] = ((const uint32_t*)ig)[o1];
    x.f[0] = ((const uint32_t*)fg)[o0], x.f[1] = ((const uint32_t*)fg)[o1];
  } else {
    x.i[0] = ((const uint16_t*)ig)[o0], x.i[1] = ((const uint16_t*)ig)[o1];
    x.f[0] = ((const uint16_t*)fg)[o0], x.f[1] = ((const uint16_t*)fg)[o1];
  }
  return x;
}
__device__ __forceinline__ float gate_value(uint32_t raw, int dtype) {
  if (dtype == 0) return __uint_as_float(raw);
  if (dtype == 1) return bf16_bits_to_f32((uint16_t)raw);
  const uint16_t half = (uint16_t)raw;
  return (float)__builtin_bit_cast(_Float16, half);
}

struct ChunkScan {
  float b[2], a[2], cm[2], w[2];  // b; a; b + cummax(it - b); b - it
  float g, amax;                  // of the whole chunk
};
__device__ __forceinline__ ChunkScan scan_chunk(const RawGates& raw, int c, int lane, int S, int dtype_gates, int sig_gate) {
  const float NEG_INF = -__builtin_inff();
  const int t0 = c * kChunk + 2 * lane;
  float lf[2], it[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const bool in = t0 + e < S;
    const float iv = gate_value(raw.i[e], dtype_gates);
    lf[e] = in ? log_sigmoid(gate_value(raw.f[e], dtype_gates)) : 0.f;
    it[e] = !in ? NEG_INF : sig_gate ? log_sigmoid(iv) : iv;
  }
  const float pair = lf[0] + lf[1];
  const float incl = wave_incl_sum(pair);
  const float b1 = incl, b0 = (incl - pair) + lf[0];
  const float rincl = wave_rev_incl_sum(pair);
  const float suf1 = rincl - pair, suf0 = suf1 + lf[1];
  const float a0 = suf0 + it[0], a1 = suf1 + it[1];
  const float x0 = it[0] - b0, x1 = it[1] - b1;
  const float pm = wave_incl_max(fmaxf(x0, x1));
  const float pm_excl = lane_up(pm, NEG_INF);
  const float cm0 = fmaxf(pm_excl, x0), cm1 = pm;
  return {{b0, b1}, {a0, a1}, {b0 + cm0, b1 + cm1}, {b0 - it[0], b1 - it[1]}, last_lane(incl), last_lane(wave_incl_max(fmaxf(a0, a1)))};
}

// m before chunk c < 4 of a head (the recurrence m_c = max(g_c + m_{c-1}, amax_c) with its sums in the order of the pre-pass)
__device__ __forceinline__ float m_before(int c, float m_init, const float* g, const float* amax) {
  if (c == 0) return fmaxf(m_init, -__builtin_inff());
  if (c == 1) return fmaxf(m_init + g[0], amax[0]);
  if (c == 2) return fmaxf(m_init + (g[0] + g[1]), fmaxf(amax[0] + g[1], amax[1]));
  const float g12 = g[1] + g[2];
  return fmaxf(m_init + (g[0] + g12), fmaxf(amax[0] + g12, fmaxf(amax[1] + g[2], amax[2])));
}

}  // namespace mlstm
