// Within-chunk scans of the gates by one wave, two positions per lane (gates.hip has the formulas): for the gate pre-pass and for the
// kernels that make their own gate vectors.
#pragma once
#include "common.h"

namespace mlstm {

// Inclusive scan over the 64 lanes by cross-lane moves of the vector unit (inside rows of 16 lanes, then row totals): a shuffle through
// LDS takes ten times as long, and a chunk needs over twenty one after the other (8 heads of 317 positions of 256/512, short_fw with its
// own gates: 14.05 us by shuffles, 13.5 so; 512 heads of 64 162.8, 153.3).  `outside`: what a lane without a source sees (nothing is done there: op(outside, x) = x).
template <typename Op>
__device__ __forceinline__ float wave_incl_scan(float x, Op op, float outside) {
#define MLSTM_DPP_STEP(ctrl, rows)                                                                                                 \
  {                                                                                                                                \
    const float y = __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(outside), __float_as_uint(x), ctrl, rows, 0xf, false)); \
    x = op(y, x);                                                                                                                  \
  }
  MLSTM_DPP_STEP(0x111, 0xf)  // row_shr:1, 2, 4, 8
  MLSTM_DPP_STEP(0x112, 0xf)
  MLSTM_DPP_STEP(0x114, 0xf)
  MLSTM_DPP_STEP(0x118, 0xf)
  MLSTM_DPP_STEP(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
  MLSTM_DPP_STEP(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef MLSTM_DPP_STEP
  return x;
}
template <typename Op>
__device__ __forceinline__ float wave_rev_incl_scan(float x, Op op, float outside) {  // over the lanes from this one on
  return __shfl_xor(wave_incl_scan(__shfl_xor(x, 63), op, outside), 63);
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
  auto add = [](float a, float b) { return a + b; };
  auto mx = [](float a, float b) { return fmaxf(a, b); };
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
  const float incl = wave_incl_scan(pair, add, 0.f);
  const float b1 = incl, b0 = (incl - pair) + lf[0];
  const float rincl = wave_rev_incl_scan(pair, add, 0.f);
  const float suf1 = rincl - pair, suf0 = suf1 + lf[1];
  const float a0 = suf0 + it[0], a1 = suf1 + it[1];
  const float x0 = it[0] - b0, x1 = it[1] - b1;
  const float pm = wave_incl_scan(fmaxf(x0, x1), mx, NEG_INF);
  float pm_excl = __shfl_up(pm, 1);
  if (lane == 0) pm_excl = NEG_INF;
  const float cm0 = fmaxf(pm_excl, x0), cm1 = pm;
  return {{b0, b1}, {a0, a1}, {b0 + cm0, b1 + cm1}, {b0 - it[0], b1 - it[1]}, last_lane(incl), last_lane(wave_incl_scan(fmaxf(a0, a1), mx, NEG_INF))};
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
