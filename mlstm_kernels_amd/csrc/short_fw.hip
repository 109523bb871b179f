// Forward of short sequences (up to 512 positions) without a backward: prompts.
//
//   H[t]    = (cs_t C0^T q_t + sum_{j <= t} P[t][j] v_j) / (normaliser_t + eps),
//   P[t][j] = (q_t . k_j) / sqrt(DHQK) * exp(u_t - w_j + G)
//   C_c     = gbar_c C_{c-1} + sum_{j in c} abar_j k_j v_j^T,   n_c = gbar_c n_{c-1} + sum_{j in c} abar_j k_j
//
// with the gate vectors of gates.hip, which few workgroups make themselves (short_fw_own_gates; G: the decay of the chunks between those of j and t; cs_t: bbar_t / sqrt(DHQK), C0 decayed
// over the chunks in front of t's).  Where the whole sequence is one
// group of source chunks no chunk state is needed: H takes all keys as score blocks, and the last state is one product over all
// positions.  Neither waits for the other, so ONE launch holds the workgroups of both:
//   * H: 64 positions x CW value columns of a (batch, head).  Its eight waves take tiles of 16 keys in turn, two at a time, fetch
//     their K rows straight into operand registers (whole rows: one trip to memory), multiply them with the Q rows in LDS and
//     write the gated tiles to LDS as 16-bit values; then V goes through LDS in batches of 256 keys, all of it requested at the
//     start.  An initial state (INIT) goes through LDS before it, 64 of its rows at a time, with the Q rows in the place of P.
//     Everything is requested as early as its registers allow and in the order of its use, Q by all waves before any K (the
//     requests of a CU are served in order), and unconditionally (NSL slabs of 64 positions, past the end the last row again: a
//     request under a branch makes the compiler wait for all of them at the first use of any).  K in operands of 16 x 32: four
//     lanes a row, 64 bytes of it in one request; of 32 x 16 two lanes and 32 bytes, at half the rate.
//   * C: a tile of RT x WT of the state.  All rows are requested at the start as well; V is scaled in fp32 and split into a 16-bit
//     head and a 16-bit remainder, two products per block, as in the scan.
// What bounds it: latency, four trips to memory or LDS in a row and the matrix work of one workgroup.  The streaming kernels
// take this in three launches (gates, a scan of up to four chunks that run twice, H from the chunk states), each with most of
// the chip idle.  us for all launches, streaming kernels / gates and this, the same rows again and again: 8 heads of 256/512, 128
// positions 27.5 / 11.8, 317 36.5 / 16.8, 512 36.5 / 27.9, 317 from a state 37.3 / 20.4; 16 heads of 128/256, 317 33.2 / 14.9.
// Rows that no cache holds: 28.7 / 13.4, 39.3 / 19.0, 39.0 / 30.7; 36.2 / 18.0.  (The gates in a launch of their own in all of these.)
#include "common.h"
#include "gate_scan.h"
#include "kernels.h"

namespace mlstm {
namespace {
constexpr int kShortThreads = 512;

template <int DQ, int CW, bool INIT>
struct ShortLds {
  // H: [Q rows, then (INIT: behind them) slabs of V | P | w | row sums, INIT: q . n0 | 1 / normaliser | OWN: b,
  // b + cummax(it - b) of the positions, decay and largest weight of every chunk | INIT: n0, cs, decay]
  static constexpr int QS = DQ + 8, VS = CW + 32;
  static constexpr int NBT = INIT ? 2 : 4;  // slabs of V at a time
  static constexpr int kFront = INIT ? 64 * QS + NBT * 64 * VS : (64 * QS > NBT * 64 * VS ? 64 * QS : NBT * 64 * VS);
  static constexpr int RT = DQ % 128 == 0 ? 128 : 64, WT = CW;  // state tile
  static constexpr int XS = RT + 32, YS = WT + 32;
  static size_t bytes(int nt, bool with_c) {
    const size_t h = (size_t)kFront * 2 + (size_t)64 * (64 * nt + 8) * 2 + kShortMax * 4 + 9 * 64 * 4 + 3 * 64 * 4 + 8 * 4 + (INIT ? (DQ + 65) * 4 : 0);
    // C: [K slab | head of V | remainder of V | abar | abar as an operand | OWN: decay, largest weight of every chunk]
    const size_t c = (size_t)64 * (XS + 2 * YS) * 2 + kShortMax * 4 + kShortMax * 3 * 2 + 8 * 4;
    return with_c && c > h ? c : h;
  }
};

// OWN: few workgroups.  Each scans the gates of its head (its waves a chunk each, while the rows are on their way), and H and the last
// state are written through the caches: what lies in the L2s at the end goes to memory while the next launch waits for it.  us, plain /
// write-through: 8 heads of 256/512, 317 positions 13.5 / 12.9, 512 26.4 / 25.5; 32 heads of 64 13.7 / 12.2; 4 heads of 512/1024, 300 23.8 /
// 22.8.  (With more it gains as much up to some 100 MB, but for 384 heads of 64 positions from a state, 192 MB of it, 169.2 / 171.2; chosen
// in the kernel it costs 512 heads of 64 124 / 133.)
template <int DQ, int CW, int NSL, bool F16, bool INIT, bool OWN>
__device__ __forceinline__ void short_h(const ShortFwArgs& a, int item, unsigned char* smem) {
  using L = ShortLds<DQ, CW, INIT>;
  constexpr int QS = L::QS, VS = L::VS;
  constexpr int NF = DQ / 32 < 8 ? DQ / 32 : 8;  // operands of a tile of K that are fetched at once
  constexpr int NGK = DQ / 32 / NF;              // ... so many times
  constexpr int QV = DQ / 64, VV = CW / 64;        // 16-byte pieces per thread: Q rows, a slab of V
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int S = a.S, DHHV = a.DHHV, NC = a.NC, nt = (S + 63) / 64, ng = DHHV / CW;
  const int g = item % ng, tq = nt - 1 - (item / ng) % nt, bh = item / (ng * nt);  // the longest first
  const int t0 = 64 * tq, c = t0 / kChunk;
  const int PSS = 64 * nt + 8;
  uint16_t* const Qs = (uint16_t*)smem;
  uint16_t* const Vs = INIT ? Qs + 64 * QS : Qs;  // (without a state Q is done with before V comes)
  uint16_t* const Ps = Qs + L::kFront;
  float* const wv = (float*)(Ps + 64 * PSS);
  float* const rows = wv + kShortMax;  // [8 waves][64], INIT: q . n0 [64]
  float* const inv = rows + 9 * 64;
  float* const bv = inv + 64;    // OWN: [2][64]
  float* const gch = bv + 128;   // OWN: [2][4]
  float* const nv = gch + 8;     // INIT: n0
  float* const csv = nv + DQ;    // INIT: cs_t, decay of the initial state up to this chunk
  const size_t Sp = (size_t)NC * kChunk, gofs = (size_t)bh * Sp;
  const uint16_t* const Qg = a.Q + (size_t)bh * S * DQ;
  const uint16_t* const Kg = a.K + (size_t)bh * S * DQ;
  const uint16_t* const Vg = a.V + (size_t)bh * S * DHHV + g * CW;
  const int n_kt = min(4 * tq + 4, (S + 15) / 16);  // tiles of 16 keys
  const int n_sl = tq + 1;                          // slabs of 64 keys

  // ---- everything this workgroup needs is requested here, the gates of a chunk by each wave first
  const int gc = min(wave, NC - 1);
  RawGates raw;
  if constexpr (OWN) raw = load_gates(a.ig, a.fg, bh, gc, lane, S, a.dtype_gates);
  u32x4 qr[QV];
#pragma unroll
  for (int x = 0; x < QV; ++x) {
    const int idx = tid + x * kShortThreads, row = idx / (DQ / 8), u = idx % (DQ / 8);
    qr[x] = *(const u32x4*)(Qg + (size_t)min(t0 + row, S - 1) * DQ + u * 8);
  }
  const int l16 = lane & 15, lq = lane >> 4;
  // (the gate vectors cover whole chunks: positions past the end have w = infinity, a factor of zero)
  float w_own = 0.f, mc = 0.f, m_init = 0.f, un[4], gr[kShortMax / kChunk];
  if constexpr (OWN) {
    if (!a.sig_gate && a.m0 != nullptr) m_init = a.m0[bh];
  } else {
    w_own = a.g.w[gofs + min(tid, (int)Sp - 1)];
#pragma unroll
    for (int tc = 0; tc < 4; ++tc) un[tc] = a.g.u[gofs + t0 + 16 * tc + l16];
    mc = a.g.mcomb[gofs + t0 + (tid & 63)];
#pragma unroll
    for (int y = 0; y < kShortMax / kChunk; ++y) gr[y] = a.g.graw[(size_t)bh * NC + min(y, NC - 1)];
  }
  __syncthreads();
  // unit x of a wave: tiles wave + 16 y and wave + 16 y + 8 (y = x / NGK), operands NF (x % NGK) .. of their rows
  Frag k0[2][NF], k1[2][NF];
  const int n_units = NGK * ((wave < n_kt ? 1 : 0) + (wave + 16 < n_kt ? 1 : 0));
  auto fetch = [&](Frag (&f)[2][NF], int x) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int kt = wave + 16 * (x / NGK) + 8 * e;
      const uint16_t* const p = Kg + (size_t)min(16 * kt + l16, S - 1) * DQ + (x % NGK) * (NF * 32) + 8 * lq;
#pragma unroll
      for (int ks = 0; ks < NF; ++ks) f[e][ks].u = *(const uint4*)(p + 32 * ks);
    }
  };
  fetch(k0, 0);

  if constexpr (OWN) {  // the scans of a chunk by each wave, while the rows are on their way
    const ChunkScan cs = scan_chunk(raw, gc, lane, S, a.dtype_gates, a.sig_gate);
    if (wave < NC) {
      *(float2*)(wv + kChunk * wave + 2 * lane) = make_float2(cs.w[0], cs.w[1]);
      if (wave == c && lane / 32 == tq % 2) {
        *(float2*)(bv + 2 * r) = make_float2(cs.b[0], cs.b[1]);
        *(float2*)(bv + 64 + 2 * r) = make_float2(cs.cm[0], cs.cm[1]);
      }
      if (lane == 0) gch[wave] = cs.g, gch[4 + wave] = cs.amax;
    }
  }
#pragma unroll
  for (int x = 0; x < QV; ++x) {
    const int idx = tid + x * kShortThreads, row = idx / (DQ / 8), u = idx % (DQ / 8);
    *(u32x4*)(Qs + row * QS + u * 8) = qr[x];
  }
  if constexpr (!OWN) wv[tid] = w_own;
  if constexpr (INIT) {
    if (tid < DQ) nv[tid] = a.use_nrow ? a.n_init[(size_t)bh * DQ + tid] : 0.f;
    if constexpr (!OWN) {
      if (tid < 64) csv[tid] = a.g.bbar[gofs + t0 + tid] * a.qk_scale;
      if (tid == 64) {
        float gsum = 0.f;
        for (int y = 0; y < c; ++y) gsum += a.g.graw[(size_t)bh * NC + y];
        const float* const mst = a.g.mstates + (size_t)bh * (NC + 1);
        csv[64] = c > 0 ? __expf(gsum + mst[0] - mst[c]) : 1.f;
      }
    }
  }
  __syncthreads();
  u32x4 vr[NSL][VV];
#pragma unroll
  for (int s = 0; s < NSL; ++s)
#pragma unroll
    for (int x = 0; x < VV; ++x) {
      const int idx = tid + x * kShortThreads, row = idx / (CW / 8), u = idx % (CW / 8);
      vr[s][x] = *(const u32x4*)(Vg + (size_t)min(64 * s + row, S - 1) * DHHV + u * 8);
    }

  float mp = 0.f;  // OWN: m before this chunk
  auto m_at = [&](int t) { return a.sig_gate ? 0.f : fmaxf(bv[t] + mp, bv[64 + t]); };
  if constexpr (OWN) {
#pragma unroll
    for (int y = 0; y < kShortMax / kChunk; ++y) gr[y] = gch[y];  // (those of chunks past the end are not used)
    if (!a.sig_gate) mp = m_before(c, m_init, gch, gch + 4);
#pragma unroll
    for (int tc = 0; tc < 4; ++tc) un[tc] = bv[16 * tc + l16] - m_at(16 * tc + l16);
    mc = m_at(lane);
    if (a.m_last != nullptr && g == 0 && tq == nt - 1 && tid == 0) a.m_last[bh] = a.sig_gate ? 0.f : fmaxf(mp + gch[c], gch[4 + c]);
  }

  // The state takes its decay up to this chunk in fp32, in front of its rounding: one beyond the range of float16 that has decayed
  // into it is finite where it is seen there.
  float pre = 1.f;
  if constexpr (INIT) {
    auto cs_at = [&](int t) { return OWN ? expf(bv[t] + mp - m_at(t)) * a.qk_scale : csv[t]; };
    if constexpr (OWN) {
      float gsum = 0.f;
#pragma unroll
      for (int y = 0; y < kShortMax / kChunk; ++y) gsum += y < c ? gr[y] : 0.f;
      if (c > 0) pre = __expf(gsum + (a.sig_gate ? 0.f : m_before(0, m_init, gch, gch + 4)) - mp);
      if (tid < 64) csv[tid] = cs_at(tid);
    } else {
      pre = csv[64];
    }
    // q_t . n0, eight threads per position
    const int t = tid >> 3, part = tid & 7;
    float dot = 0.f;
#pragma unroll
    for (int d = 0; d < DQ / 8; d += 4) {
      const uint2 qv = *(const uint2*)(Qs + t * QS + part * (DQ / 8) + d);
      const float4 n4 = *(const float4*)(nv + part * (DQ / 8) + d);
      dot += lo2<F16>(qv.x) * n4.x + hi2<F16>(qv.x) * n4.y + lo2<F16>(qv.y) * n4.z + hi2<F16>(qv.y) * n4.w;
    }
    dot += __shfl_xor(dot, 1);
    dot += __shfl_xor(dot, 2);
    dot += __shfl_xor(dot, 4);
    if (part == 0) rows[8 * 64 + t] = cs_at(t) * pre * dot;
  }
  // ---- scores of this wave's tiles, gated into P
  {
    const float lsc = __log2f(a.qk_scale);
    float rsum[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4 sacc[2][4];
    auto unit = [&](const Frag (&f)[2][NF], int x) __attribute__((always_inline)) {
      const int gk = x % NGK;
      if (gk == 0) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int tc = 0; tc < 4; ++tc) sacc[e][tc] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int ks = 0; ks < NF; ++ks)
#pragma unroll
        for (int tc = 0; tc < 4; ++tc) {
          Frag B;
          B.u = *(const uint4*)(Qs + (16 * tc + l16) * QS + (gk * NF + ks) * 32 + 8 * lq);
#pragma unroll
          for (int e = 0; e < 2; ++e) mfma16<F16>(sacc[e][tc], f[e][ks], B);  // rows: keys, columns: positions
        }
      if (gk == NGK - 1) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int kt = wave + 16 * (x / NGK) + 8 * e;
          if (kt < n_kt) {
            float G = 0.f;  // decay of the chunks between the keys' and the positions'
#pragma unroll
            for (int y = 0; y < kShortMax / kChunk; ++y) G += y >= kt / 8 && y < c ? gr[y] : 0.f;
            const float4 wj = *(const float4*)(wv + 16 * kt + 4 * lq);
            const float w4[4] = {wj.x, wj.y, wj.z, wj.w};
#pragma unroll
            for (int tc = 0; tc < 4; ++tc) {
              const int diag = 4 * tq + tc;  // tile of the positions themselves
              if (kt <= (diag | 1)) {        // (P is read in blocks of 32 positions)
                float p[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const float e2 = __builtin_amdgcn_exp2f(__builtin_fmaf(un[tc] + G - w4[q], 1.4426950408889634f, lsc));
                  p[q] = kt < diag || (kt == diag && 4 * lq + q <= l16) ? sacc[e][tc][q] * e2 : 0.f;
                  rsum[tc] += p[q];
                }
                *(uint2*)(Ps + (16 * tc + l16) * PSS + 16 * kt + 4 * lq) = make_uint2(pack2<F16>(p[0], p[1]), pack2<F16>(p[2], p[3]));
              }
            }
          }
        }
      }
    };
    for (int x = 0; x < n_units; x += 2) {
      if (x + 1 < n_units) fetch(k1, x + 1);
      unit(k0, x);
      if (x + 1 < n_units) {
        if (x + 2 < n_units) fetch(k0, x + 2);
        unit(k1, x + 1);
      }
    }
#pragma unroll
    for (int tc = 0; tc < 4; ++tc) {
      float tot = rsum[tc] + __shfl_xor(rsum[tc], 16);
      tot += __shfl_xor(tot, 32);
      if (lq == 0) rows[wave * 64 + 16 * tc + l16] = tot;
    }
  }
  __syncthreads();

  // ---- denominators; Out^T += V^T P over the keys
  if (tid < 64) {
    float iv = 1.f, nmax = 1.f;
    if (a.use_nrow) {
      float den = INIT ? rows[8 * 64 + tid] : 0.f;
#pragma unroll
      for (int y = 0; y < 8; ++y) den += rows[y * 64 + tid];
      nmax = fmaxf(fabsf(den), a.sig_gate ? 1.f : __expf(-mc));
      iv = 1.f / (nmax + a.eps);
    }
    inv[tid] = iv;
    if (g == 0 && t0 + tid < S) {
      const size_t tg = (size_t)bh * S + t0 + tid;
      if (a.n_out != nullptr) a.n_out[tg] = nmax;
      if (a.m_out != nullptr) a.m_out[tg] = mc;
    }
  }
  constexpr int NCB = CW / 32;  // column blocks of 32: one and 32 positions for each wave (CW = 64: for four of them)
  const int cb = wave % NCB, tb = wave / NCB;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  auto store_slab = [&](int s, const u32x4 (&v)[VV]) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < VV; ++x) {
      const int idx = tid + x * kShortThreads, row = idx / (CW / 8), u = idx % (CW / 8);
      const u32x4 none = {0u, 0u, 0u, 0u};
      *(u32x4*)(Vs + (s % L::NBT) * (64 * VS) + row * VS + u * 8) = 64 * s + row < S ? v[x] : none;
    }
  };
  const int q16 = (lane >> 4) & 1, i16 = lane & 15;
  const int krow = 8 * h + (i16 >> 2), ncol = 16 * q16 + 4 * (i16 & 3);
  if constexpr (INIT) {
    // Out^T = C0^T Q^T over the head dimension, 64 rows of C0 at a time, rounded like every state that is multiplied
    const float* const Cg = a.init + (size_t)bh * DQ * DHHV + g * CW;
    f32x4 cr[2][VV][2];
    auto fetch_c = [&](f32x4 (&x)[VV][2], int s) __attribute__((always_inline)) {
#pragma unroll
      for (int y = 0; y < VV; ++y) {
        const int idx = tid + y * kShortThreads, row = idx / (CW / 8), u = idx % (CW / 8);
        const float* const p = Cg + (size_t)(64 * s + row) * DHHV + u * 8;
        x[y][0] = *(const f32x4*)p;
        x[y][1] = *(const f32x4*)(p + 4);
      }
    };
    fetch_c(cr[0], 0);
#pragma unroll
    for (int s = 0; s < DQ / 64; ++s) {
      if (s + 1 < DQ / 64) fetch_c(cr[(s + 1) & 1], s + 1);
      uint16_t* const slab = Vs + (s & 1) * (64 * VS);
#pragma unroll
      for (int y = 0; y < VV; ++y) {
        const int idx = tid + y * kShortThreads, row = idx / (CW / 8), u = idx % (CW / 8);
        const f32x4 lo = cr[s & 1][y][0] * pre, hi = cr[s & 1][y][1] * pre;
        *(uint4*)(slab + row * VS + u * 8) = make_uint4(pack2<F16>(lo[0], lo[1]), pack2<F16>(lo[2], lo[3]), pack2<F16>(hi[0], hi[1]), pack2<F16>(hi[2], hi[3]));
      }
      __syncthreads();
      if (tb < 2) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          Frag A, B;
          const uint16_t* const p = slab + (16 * kk + krow) * VS + 32 * cb + ncol;
          A.d[0] = lds_read_tr16(p);
          A.d[1] = lds_read_tr16(p + 4 * VS);
          B.u = *(const uint4*)(Qs + (32 * tb + r) * QS + 64 * s + 16 * kk + 8 * h);
          mfma32<F16>(acc, A, B);
        }
      }
    }
    if (tb < 2) acc *= csv[32 * tb + r];
  }
#pragma unroll
  for (int s0 = 0; s0 < NSL; s0 += L::NBT)
    if (s0 < n_sl) {
      if (INIT || s0 > 0) __syncthreads();  // (what lies there has been read)
#pragma unroll
      for (int s = s0; s < s0 + L::NBT && s < NSL; ++s)
        if (s < n_sl) store_slab(s, vr[s]);
      __syncthreads();
      if (tb < 2) {
        // key blocks above the diagonal are left out: zero times a NaN or infinity in V would be NaN.  So are those past the last
        // tile of keys, where P holds what LDS held before (V is zero there, but that may be a NaN)
        const int kk_end = min(min(4 * (s0 + L::NBT), n_kt), 4 * tq + 2 * tb + 2);
#pragma unroll 4
        for (int kk = 4 * s0; kk < kk_end; ++kk) {
          Frag A, B;
          const uint16_t* const p = Vs + (16 * (kk - 4 * s0) + krow) * VS + 32 * cb + ncol;
          A.d[0] = lds_read_tr16(p);
          A.d[1] = lds_read_tr16(p + 4 * VS);
          B.u = *(const uint4*)(Ps + (32 * tb + r) * PSS + 16 * kk + 8 * h);
          mfma32<F16>(acc, A, B);  // rows: value columns, columns: positions
        }
      }
    }
  __syncthreads();
  // ---- rows out through LDS
  constexpr int OS = CW + 8;
  uint16_t* const Os = Vs;
  if (tb < 2) {
    const float iv = inv[32 * tb + r];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *(uint2*)(Os + (32 * tb + r) * OS + 32 * cb + 8 * g4 + 4 * h) =
          make_uint2(pack2<F16>(acc[4 * g4] * iv, acc[4 * g4 + 1] * iv), pack2<F16>(acc[4 * g4 + 2] * iv, acc[4 * g4 + 3] * iv));
  }
  __syncthreads();
  uint16_t* const Og = a.Out + ((size_t)bh * S + t0) * DHHV + g * CW;
#pragma unroll
  for (int x = 0; x < VV; ++x) {
    const int idx = tid + x * kShortThreads, row = idx / (CW / 8), u = idx % (CW / 8);
    if (t0 + row < S) {
      const u32x4 x4 = *(const u32x4*)(Os + row * OS + u * 8);
      if constexpr (OWN) store_write_through(Og, 64 * (uint32_t)DHHV * 2, (row * (uint32_t)DHHV + u * 8) * 2, x4);
      else *(u32x4*)(Og + (size_t)row * DHHV + u * 8) = x4;
    }
  }
}

template <int DQ, int CW, int NSL, bool F16, bool INIT, bool OWN>
__device__ __forceinline__ void short_c(const ShortFwArgs& a, int item, unsigned char* smem) {
  using L = ShortLds<DQ, CW, INIT>;
  constexpr int RT = L::RT, WT = L::WT, XS = L::XS, YS = L::YS;
  constexpr int XV = RT / 64, YV = WT / 64;          // 16-byte pieces per thread and slab
  constexpr int NRB = RT / 32, NCB = WT / 32;        // blocks of 32 x 32
  constexpr int NBW = NRB * NCB > 8 ? NRB * NCB / 8 : 1;  // blocks per wave, side by side
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int S = a.S, DHHV = a.DHHV, NC = a.NC;
  constexpr int nx = DQ / RT;
  const int ny = DHHV / WT;
  const int bx = item % nx, by = (item / nx) % ny, bh = item / (nx * ny);
  uint16_t* const Xs = (uint16_t*)smem;
  uint16_t* const Yh = Xs + 64 * XS;
  uint16_t* const Yl = Yh + 64 * YS;
  float* const wt = (float*)(Yl + 64 * YS);
  uint16_t* const nB = (uint16_t*)(wt + kShortMax);  // [position / 8][3][8]
  float* const gch = (float*)(nB + kShortMax * 3);   // OWN: [2][4]
  const uint16_t* const Kg = a.K + (size_t)bh * S * DQ + bx * RT;
  const uint16_t* const Vg = a.V + (size_t)bh * S * DHHV + by * WT;
  const int n_sl = (S + 63) / 64;
  auto weight = [&](int t, float w) {
    wt[t] = w;
    // n as in the scan: the weights, split exactly into three 16-bit parts, are three columns of one more operand
    uint16_t* const dst = nB + (t >> 3) * 24 + (t & 7);
    const uint16_t p0 = f32_to_elem<F16>(w);
    const float r1 = w - elem_to_f32<F16>(p0);
    const uint16_t p1 = f32_to_elem<F16>(r1);
    dst[0] = p0;
    dst[8] = p1;
    dst[16] = f32_to_elem<F16>(r1 - elem_to_f32<F16>(p1));
  };
  // (the decay of later chunks is left to the sums: the largest weight of a chunk is one, and one times v has no remainder)
  float gb[kShortMax / kChunk];
  const int gc = min(wave, NC - 1);
  RawGates raw;
  float m_init = 0.f;
  if constexpr (OWN) {
    raw = load_gates(a.ig, a.fg, bh, gc, lane, S, a.dtype_gates);
    if (!a.sig_gate && a.m0 != nullptr) m_init = a.m0[bh];
  } else {
    const float ab = a.g.abar[(size_t)bh * NC * kChunk + min(tid, NC * kChunk - 1)];
    weight(tid, tid < S ? ab : 0.f);
#pragma unroll
    for (int y = 0; y < kShortMax / kChunk; ++y) gb[y] = a.g.gbar[(size_t)bh * NC + min(y, NC - 1)];
  }
  u32x4 xr[NSL][XV], yr[NSL][YV];
#pragma unroll
  for (int s = 0; s < NSL; ++s) {
#pragma unroll
    for (int x = 0; x < XV; ++x) {
      const int idx = tid + x * kShortThreads, row = idx / (RT / 8), u = idx % (RT / 8);
      xr[s][x] = *(const u32x4*)(Kg + (size_t)min(64 * s + row, S - 1) * DQ + u * 8);
    }
#pragma unroll
    for (int x = 0; x < YV; ++x) {
      const int idx = tid + x * kShortThreads, row = idx / (WT / 8), u = idx % (WT / 8);
      yr[s][x] = *(const u32x4*)(Vg + (size_t)min(64 * s + row, S - 1) * DHHV + u * 8);
    }
  }
  if constexpr (OWN) {  // the scans of a chunk by each wave, while the rows are on their way
    const ChunkScan cs = scan_chunk(raw, gc, lane, S, a.dtype_gates, a.sig_gate);
    if (lane == 0 && wave < NC) gch[wave] = cs.g, gch[4 + wave] = cs.amax;
    __syncthreads();
#pragma unroll
    for (int y = 0; y < kShortMax / kChunk; ++y) {
      gb[y] = 1.f;
      if (y < NC) {
        const float mp = a.sig_gate ? 0.f : m_before(y, m_init, gch, gch + 4);
        const float mn = a.sig_gate ? 0.f : fmaxf(mp + gch[y], gch[4 + y]);
        gb[y] = expf(gch[y] + mp - mn);
        if (wave == y) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int t = kChunk * y + 2 * lane + e;
            weight(t, t < S ? expf(cs.a[e] - mn) : 0.f);
          }
        }
      }
    }
  }
  const int rb = wave % NRB, cb0 = wave / NRB * NBW;
  const bool busy = cb0 < NCB;
  f32x16 acc[NBW], rest[NBW];  // sums of the heads and of the remainders: a remainder does not cost the large sum a rounding
#pragma unroll
  for (int b = 0; b < NBW; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[b][i] = rest[b][i] = 0.f;
  const bool with_n = a.n_final != nullptr && by == 0 && cb0 == 0;  // this wave carries n of its 32 rows
  f32x16 accn;
#pragma unroll
  for (int i = 0; i < 16; ++i) accn[i] = 0.f;
  if constexpr (INIT) {
    if (busy) {
#pragma unroll
      for (int b = 0; b < NBW; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int d = bx * RT + 32 * rb + 8 * (i / 4) + 4 * h + (i % 4);
          acc[b][i] = a.init[((size_t)bh * DQ + d) * DHHV + by * WT + 32 * (cb0 + b) + r];
        }
    }
    if (with_n && r == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) accn[i] = a.n_init[(size_t)bh * DQ + bx * RT + 32 * rb + 8 * (i / 4) + 4 * h + (i % 4)];
    }
  }
  const int q16 = (lane >> 4) & 1, i16 = lane & 15;
  const int krow = 8 * h + (i16 >> 2), ncol = 16 * q16 + 4 * (i16 & 3);
#pragma unroll
  for (int s = 0; s < NSL; ++s)
    if (s < n_sl) {
      __syncthreads();
#pragma unroll
      for (int x = 0; x < XV; ++x) {
        const int idx = tid + x * kShortThreads, row = idx / (RT / 8), u = idx % (RT / 8);
        *(u32x4*)(Xs + row * XS + u * 8) = xr[s][x];
      }
#pragma unroll
      for (int x = 0; x < YV; ++x) {
        const int idx = tid + x * kShortThreads, row = idx / (WT / 8), u = idx % (WT / 8);
        const float w = wt[64 * s + row];
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float e0 = lo2<F16>(yr[s][x][e]) * w, e1 = hi2<F16>(yr[s][x][e]) * w;
          // (head and remainder of the same fp32 product: to float16 it may be converted and multiplied in one step)
          if constexpr (F16) asm("" : "+v"(e0), "+v"(e1));
          hi[e] = pack2<F16>(e0, e1);
          lo[e] = pack2<F16>(e0 - lo2<F16>(hi[e]), e1 - hi2<F16>(hi[e]));
        }
        *(uint4*)(Yh + row * YS + u * 8) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *(uint4*)(Yl + row * YS + u * 8) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      }
      __syncthreads();
      if (s % 2 == 0 && (INIT || s > 0)) {
#pragma unroll
        for (int b = 0; b < NBW; ++b) {
          acc[b] *= gb[s / 2];
          rest[b] *= gb[s / 2];
        }
        accn *= gb[s / 2];
      }
      if (busy) {
#pragma unroll
        for (int js = 0; js < 4; ++js) {
          Frag A;
          const uint16_t* const p = Xs + (16 * js + krow) * XS + 32 * rb + ncol;
          A.d[0] = lds_read_tr16(p);
          A.d[1] = lds_read_tr16(p + 4 * XS);
#pragma unroll
          for (int b = 0; b < NBW; ++b) {
            const int o = (16 * js + krow) * YS + 32 * (cb0 + b) + ncol;
            Frag Bh, Bl;
            Bh.d[0] = lds_read_tr16(Yh + o);
            Bh.d[1] = lds_read_tr16(Yh + o + 4 * YS);
            Bl.d[0] = lds_read_tr16(Yl + o);
            Bl.d[1] = lds_read_tr16(Yl + o + 4 * YS);
            mfma32<F16>(acc[b], A, Bh);
            mfma32<F16>(rest[b], A, Bl);
          }
          if (with_n) {
            Frag Bn;
            Bn.u = *(const uint4*)(nB + (8 * s + 2 * js + h) * 24 + min(r, 2) * 8);
            if (r >= 3) Bn.u = make_uint4(0u, 0u, 0u, 0u);
            mfma32<F16>(accn, A, Bn);
          }
        }
      }
    }
  if (busy) {
#pragma unroll
    for (int b = 0; b < NBW; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = bx * RT + 32 * rb + 8 * (i / 4) + 4 * h + (i % 4);
        const float x = acc[b][i] + rest[b][i];
        if constexpr (OWN) {
          store_write_through(a.final_out + (size_t)bh * DQ * DHHV, DQ * (uint32_t)DHHV * 4, (uint32_t)(d * DHHV + by * WT + 32 * (cb0 + b) + r) * 4, __float_as_uint(x));
        } else {
          a.final_out[((size_t)bh * DQ + d) * DHHV + by * WT + 32 * (cb0 + b) + r] = x;
        }
      }
  }
  if (with_n) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float x = accn[i];
      const float sum = __shfl(x, 32 * h) + __shfl(x, 32 * h + 1) + __shfl(x, 32 * h + 2);
      if (r == 0) a.n_final[(size_t)bh * DQ + bx * RT + 32 * rb + 8 * (i / 4) + 4 * h + (i % 4)] = sum;
    }
  }
}

}  // namespace

template <int DQ, int CW, int NSL, bool F16, bool INIT, bool OWN>
__global__ __launch_bounds__(kShortThreads) void short_fw_kernel(ShortFwArgs a, int n_h, int n_c) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // consecutive items (of one head) share an XCD and the head's rows in its L2
  int b = blockIdx.x;
  const bool is_h = b < n_h;
  if (!is_h) b -= n_h;
  const int n = is_h ? n_h : n_c;
  if (n_h % 8 == 0 && n % 8 == 0) b = (b % 8) * (n / 8) + b / 8;
  if (is_h) short_h<DQ, CW, NSL, F16, INIT, OWN>(a, b, smem_raw);
  else short_c<DQ, CW, NSL, F16, INIT, OWN>(a, b, smem_raw);
}

namespace {
template <int DQ, int CW, int NSL, bool F16, bool INIT, bool OWN>
const char* launch_short_t(const ShortFwArgs& a, int BH, hipStream_t stream) {
  using L = ShortLds<DQ, CW, INIT>;
  const int nt = (a.S + 63) / 64;
  const long long n_h = (long long)BH * nt * (a.DHHV / CW);
  const long long n_c = a.final_out == nullptr ? 0 : (long long)BH * (DQ / L::RT) * (a.DHHV / L::WT);
  if (n_h + n_c >= (1ll << 31)) return "short_fw: too many workgroups";
  const size_t smem = L::bytes(nt, n_c > 0);
  if (smem > 160 * 1024) return "short_fw: too long for one CU's LDS";
  static LdsLimit lds;
  if (!lds.allow((const void*)short_fw_kernel<DQ, CW, NSL, F16, INIT, OWN>, smem)) return "short_fw: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((short_fw_kernel<DQ, CW, NSL, F16, INIT, OWN>), dim3((unsigned)(n_h + n_c)), dim3(kShortThreads), smem, stream, a, (int)n_h, (int)n_c);
  return nullptr;
}
template <int DQ, int CW, int NSL, bool F16, bool INIT>
const char* launch_short_g(const ShortFwArgs& a, int BH, hipStream_t stream) {
  return a.own_gates ? launch_short_t<DQ, CW, NSL, F16, INIT, true>(a, BH, stream) : launch_short_t<DQ, CW, NSL, F16, INIT, false>(a, BH, stream);
}
template <int DQ, int CW, int NSL>
const char* launch_short_c(const ShortFwArgs& a, int BH, hipStream_t stream) {
  if (a.init != nullptr) {
    // (the Q rows of 512 beside the V slabs and more than five score tiles do not fit the LDS: no instance)
    if constexpr (DQ == 512 && NSL > 5) return "short_fw: too long for one CU's LDS";
    else return a.f16 ? launch_short_g<DQ, CW, NSL, true, true>(a, BH, stream) : launch_short_g<DQ, CW, NSL, false, true>(a, BH, stream);
  }
  return a.f16 ? launch_short_g<DQ, CW, NSL, true, false>(a, BH, stream) : launch_short_g<DQ, CW, NSL, false, false>(a, BH, stream);
}
template <int DQ, int CW>
const char* launch_short_s(const ShortFwArgs& a, int BH, hipStream_t stream) {
  // Registers and requests for as many slabs as there are, in three steps.  us, 8 heads of 256/512, gates and this / eight slabs
  // always / an instance for every number: 128 positions 11.8 / 12.9 / 11.8, 192 13.6 / 14.1 / 13.3, 317 16.8 / 17.4 / 17.0, 321 19.1 /
  // 19.1 / 18.3, 448 25.7 / 25.7 / 25.6; 16 heads of 128/256: 128 9.9 / 11.4 / 10.0, 129 12.4 / 13.1 / 11.9, 384 16.9 / 16.9 / 16.5.
  if (a.S <= 128) return launch_short_c<DQ, CW, 2>(a, BH, stream);
  return a.S <= 320 ? launch_short_c<DQ, CW, 5>(a, BH, stream) : launch_short_c<DQ, CW, 8>(a, BH, stream);
}
template <int DQ>
const char* launch_short_d(const ShortFwArgs& a, int BH, hipStream_t stream) {
  return a.DHHV % 128 == 0 ? launch_short_s<DQ, 128>(a, BH, stream) : launch_short_s<DQ, 64>(a, BH, stream);
}
}  // namespace

// Where this kernel is the faster one: a workgroup of H takes 5 to 12 us by its number of keys and a CU one at a time, so with
// many heads scan + H, which keep the memory system busy, overtake it -- the sooner the longer the sequence and the larger the
// head.  The line is drawn in positions in 64s times workgroups of H, per CU; an initial state counts as two more slabs.  us,
// gates + scan + H / gates + this, B sequences (rows no cache holds up to 128 positions, repeated calls beyond):
//  * more than 128 positions, 16.  256/512, 8 heads a sequence: 200 positions B=4 48 / 37, B=8 64 / 60, B=16 95 / 106; 317: B=1 42.9
//    / 21.5, B=4 51 / 46, B=8 73 / 79; 512: B=1 42.8 / 33.1, B=2 45 / 48, B=4 52 / 74.  128/256, 16 heads: 200 B=8 53 / 46, B=16 72 /
//    79; 512 B=2 40.6 / 39.4, B=4 49 / 60; 64/64, 8 heads: 512 B=8 37 / 30, B=16 39 / 45; 512/1024, 4 heads: 512 B=2 70 / 64, B=4 86 /
//    114.  With a state, 256/512: 200 B=4 50 / 44, B=8 66 / 77, 512 B=1 44 / 37, B=2 47 / 55.
//  * up to 128 positions in relation to the head: a head of 64 or 128 rows counts a quarter or a half, groups of 64 columns half.
//    65 to 128 positions, 12, of 128: 128/256, 16 heads, B=32 72 / 74, B=48 104 / 109; 256/256, 8 heads, B=48 88 / 82, B=64 107 /
//    115; 512/1024, 4 heads, B=24 165 / 135, B=32 145 / 162; 64/64, 8 heads, B=128 63 / 38; with a state 128/256 B=24 88 / 81, B=32
//    97 / 107, 256/256 B=24 72 / 69, B=32 85 / 92.  7 where the other side is the streaming H / dV kernel: 256/512, 8 heads, B=8 35 /
//    30, B=12 41 / 41, B=16 48.5 / 51, B=64 157 / 207; with a state B=4 34 / 24, B=8 49 / 48, B=12 59 / 67.
//    Up to 64 positions without a state there is no line (256/512 B=64 138 / 116, 512/1024 B=32 142 / 105, 256/256 B=128 174 / 125;
//    1024 heads of 64 positions with all launches, groups of 64 columns: 64/192 127 / 49, 512/448 1105 / 615, 64/960 477 / 247);
//    with one, 24 (256/256 B=128 269 / 240, 128/256 B=64 164 / 125) and 18 with the streaming kernel (256/512 B=48 170 / 168, B=64
//    213 / 222).
bool short_fw_preferred(const ShortFwArgs& a, int BH) {
  if (a.S > kShortMax || a.DHHV % 64 != 0) return false;
  if (a.DHQK != 64 && a.DHQK != 128 && a.DHQK != 256 && a.DHQK != 512) return false;
  if (a.DHQK == 512 && a.init != nullptr && a.S > 320) return false;  // LDS
  if ((uintptr_t)a.init % 16 != 0) return false;                      // (read by fours; the scan reads it one by one)
  const long long nt = (a.S + 63) / 64;
  const bool init = a.init != nullptr, wide = a.DHHV % 128 == 0;
  long long cost = BH * nt * (a.DHHV / (wide ? 128 : 64)) * (nt + (init ? 2 : 0));
  if (nt > 2) return cost <= 16ll * device_cu_count();
  if (nt == 1 && !init) return true;
  cost = cost * (a.DHQK < 256 ? a.DHQK : 256) / (wide ? 256 : 512);
  const bool streaming = a.DHQK == 256 && a.DHHV % 512 == 0;
  return cost <= (nt == 1 ? (streaming ? 18ll : 24ll) : (streaming ? 7ll : 12ll)) * device_cu_count();
}

// Whether its workgroups scan the gates themselves: each repeats the scans of its head, about a microsecond while its rows are on
// their way, and the launch in front (4 us) is left out.  The line is at three workgroups a CU.  us, with the pre-pass / without, bf16:
// 8 heads of 256/512, 64 positions 14.0 / 11.0 (of which the host takes all), 317 17.5 / 13.5, 512 28.5 / 26.4, 317 from a state
// 20.6 / 16.4; 16 heads of 317 26.0 / 24.0 (1.75 workgroups a CU), 32 of 64 15.1 / 13.8 (1.5), 128 heads of 128/256 of 100 positions 22.1 /
// 21.8 (3.0), 32 of 317 42.1 / 41.9 (3.5), 64 of 200 55.4 / 58.0 (6.0), 512 of 64 124.7 / 153.3 (24).
// (H goes out in write-through stores of 16 bytes, which take addresses that are multiples of 16.)
bool short_fw_own_gates(const ShortFwArgs& a, int BH) {
  if ((uintptr_t)a.Out % 16 != 0) return false;
  const long long cw = a.DHHV % 128 == 0 ? 128 : 64, rt = a.DHQK % 128 == 0 ? 128 : 64;
  const long long tiles = (a.S + 63) / 64 + (a.final_out == nullptr ? 0 : a.DHQK / rt);
  return BH * tiles * (a.DHHV / cw) <= 3ll * device_cu_count();
}

const char* launch_short_fw(const ShortFwArgs& a, int BH, hipStream_t stream) {
  if (a.S < 1 || a.S > kShortMax || a.NC != (a.S + kChunk - 1) / kChunk || a.DHHV % 64 != 0) return "short_fw: unsupported shape";
  if (a.n_final != nullptr && a.final_out == nullptr) return "short_fw: n_last without c_last";
  if ((uintptr_t)a.init % 16 != 0) return "short_fw: the initial state must lie at a multiple of 16 bytes";
  switch (a.DHQK) {
    case 64: return launch_short_d<64>(a, BH, stream);
    case 128: return launch_short_d<128>(a, BH, stream);
    case 256: return launch_short_d<256>(a, BH, stream);
    case 512: return launch_short_d<512>(a, BH, stream);
    default: return "short_fw: unsupported head dimension";
  }
}

}  // namespace mlstm
