// Fused recurrent decode step of the mLSTM (exponential input gate), one token per (batch, head).
//
//   m' = max(logsig(f) + m, i)          f' = exp(logsig(f) + m - m')      i' = exp(i - m')
//   C' = f' C + i' k v^T                n' = f' n + i' k
//   h  = (q/sqrt(d))^T C' / (max(|q/sqrt(d) . n'|, exp(-m')) + eps)
//
// (math of mlstm_kernels/torch/recurrent/native_step.py:69-95 in the reference; everything in fp32.)
//
// The step is a pure stream over the state C (DHQK x DHHV per head; fp32, or bfloat16 when the caller keeps its states
// in that type): one read and one write of every element, 0.75 flop per byte at fp32, so it is laid out for HBM
// bandwidth only -- no matrix cores.  A workgroup owns (b, head, slice of COLS value columns); lanes of 16 B (four fp32
// or eight bf16 columns) cover one contiguous row segment and the TY
// row groups of the workgroup walk the DHQK rows with all loads of an unrolled batch in flight before the first
// use.  The q^T C' column sums are reduced across the row groups through LDS at the end.
#include "common.h"
#include "kernels.h"

namespace mlstm {

// One 16-byte piece of a state row: four fp32 columns, or eight columns when the state is kept in bfloat16 or float16
// (the reference's dtype_state / inference_state_dtype, mlstm_kernels/torch/recurrent/triton_step.py:33,67-69).
// SBF = state dtype code: 0 float32, 1 bfloat16, 2 float16.
template <int SBF>
struct StatePiece {
  static constexpr int N = SBF ? 8 : 4;
  float x[N];
};
template <int SBF, bool NT>
__device__ __forceinline__ StatePiece<SBF> load_piece(const void* base, size_t elem) {
  StatePiece<SBF> p;
  if constexpr (SBF != 0) {
    const u32x4* src = (const u32x4*)((const uint16_t*)base + elem);
    const u32x4 raw = NT ? __builtin_nontemporal_load(src) : *src;
#pragma unroll
    for (int e = 0; e < 4; ++e) unpack_state2(raw[e], SBF, p.x[2 * e], p.x[2 * e + 1]);
  } else {
    const f32x4* src = (const f32x4*)((const float*)base + elem);
    const f32x4 raw = NT ? __builtin_nontemporal_load(src) : *src;
#pragma unroll
    for (int e = 0; e < 4; ++e) p.x[e] = raw[e];
  }
  return p;
}
// How a state is stored.  Plain: it stays in the L2s, which hand what they still hold to memory when the launch ends and the next one
// waits.  Write-through (device scope): on its way to memory at once, the lines stay readable.  Non-temporal: past the caches.
enum StoreMode { kPlain, kNonTemporal, kWriteThrough };
template <int MODE>
__device__ __forceinline__ void store16(void* head, uint32_t head_bytes, size_t ofs, u32x4 raw) {
  if constexpr (MODE == kNonTemporal) __builtin_nontemporal_store(raw, (u32x4*)((char*)head + ofs));
  else if constexpr (MODE == kWriteThrough) store_write_through(head, head_bytes, (uint32_t)ofs, raw);
  else *(u32x4*)((char*)head + ofs) = raw;
}
// (head: the state of the (batch, head), the same for all lanes)
template <int SBF, int MODE>
__device__ __forceinline__ void store_piece(void* head, uint32_t head_bytes, size_t elem, const StatePiece<SBF>& p) {
  if constexpr (SBF != 0) {
    const u32x4 raw = {pack_state2(p.x[0], p.x[1], SBF), pack_state2(p.x[2], p.x[3], SBF), pack_state2(p.x[4], p.x[5], SBF),
                       pack_state2(p.x[6], p.x[7], SBF)};
    store16<MODE>(head, head_bytes, elem * 2, raw);
  } else {
    store16<MODE>(head, head_bytes, elem * 4, u32x4{__float_as_uint(p.x[0]), __float_as_uint(p.x[1]), __float_as_uint(p.x[2]), __float_as_uint(p.x[3])});
  }
}

template <int COLS, int TY, int UNROLL, int MODE, int SBF>
__global__ __launch_bounds__((COLS / StatePiece<SBF>::N) * TY) void step_kernel(
    const void* __restrict__ q, const void* __restrict__ k, const void* __restrict__ v,
    const void* __restrict__ ig, const void* __restrict__ fg,
    const void* c_in, const void* n_in, const void* m_in,
    void* __restrict__ h, void* c_out, void* n_out, void* m_out,
    int DHQK, int DHHV, float eps, int dtype_qkv, int dtype_gates) {
  constexpr bool NONTEMPORAL = MODE == kNonTemporal;
  constexpr int VPL = StatePiece<SBF>::N;   // state columns per lane
  constexpr int TX = COLS / VPL;
  constexpr int NTH = TX * TY;
  constexpr int dtype_state = SBF;
  extern __shared__ float smem[];
  float* qs = smem;                 // [DHQK] q / sqrt(d)
  float* ik = smem + DHQK;          // [DHQK] i' * k
  float* red = smem + 2 * DHQK;     // [TY][COLS] partial column sums
  const int bh = blockIdx.y;
  const int col0 = blockIdx.x * COLS;
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;

  // Small states (the cacheable variant: few workgroups per CU, nothing else to hide the prologue behind): the
  // first batch of state rows is requested before anything else, so that the loads travel while the gates, q.n'
  // and the LDS staging below are computed (none of which they depend on).  With a large state many workgroups
  // per CU overlap each other's prologues and the extra live registers only cost occupancy (measured: 0.373 ms
  // against 0.358 ms at B = 256), so the streaming variant does not do it.
  const int col = col0 + VPL * tx;
  const bool col_ok = col < DHHV;  // DHHV % VPL == 0 is checked on the host
  const size_t cbase = (size_t)bh * DHQK * DHHV + col;
  void* const c_head = (char*)c_out + (size_t)bh * DHQK * DHHV * (SBF ? 2 : 4);
  const uint32_t c_bytes = (uint32_t)DHQK * DHHV * (SBF ? 2 : 4);  // (write-through: below 2^32 by the rule of launch_step)
  const bool have_first = !NONTEMPORAL && col_ok && ty + (UNROLL - 1) * TY < DHQK;
  StatePiece<SBF> cfirst[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    if (have_first) {
      cfirst[u] = load_piece<SBF, false>(c_in, cbase + (size_t)(ty + u * TY) * DHHV);
    } else {
#pragma unroll
      for (int e = 0; e < VPL; ++e) cfirst[u].x[e] = 0.f;
    }
  }

  const float fpre = load_scalar(fg, bh, dtype_gates);
  const float ipre = load_scalar(ig, bh, dtype_gates);
  const float m_old = load_state_scalar(m_in, bh, dtype_state);
  const float lf = log_sigmoid(fpre);
  const float m_new = fmaxf(lf + m_old, ipre);
  const float fa = expf(lf + m_old - m_new);
  const float ia = expf(ipre - m_new);
  const float scale = rsqrtf((float)DHQK);

  // q.n' over the whole head (every workgroup needs it for the denominator)
  float qn_part = 0.f;
  for (int d = tid; d < DHQK; d += NTH) {
    const size_t o = (size_t)bh * DHQK + d;
    const float qd = load_scalar(q, o, dtype_qkv) * scale;
    const float kd = load_scalar(k, o, dtype_qkv);
    const float nd = fa * load_state_scalar(n_in, o, dtype_state) + ia * kd;
    qs[d] = qd;
    ik[d] = ia * kd;
    qn_part += qd * nd;
    if (blockIdx.x == 0) store_state_scalar(n_out, o, dtype_state, nd);
  }
  qn_part = wave_sum(qn_part);
  __shared__ float wsum[(NTH + kWave - 1) / kWave];
  if ((tid & 63) == 0) wsum[tid >> 6] = qn_part;
  __syncthreads();
  float qn = 0.f;
#pragma unroll
  for (int w = 0; w < (NTH + kWave - 1) / kWave; ++w) qn += wsum[w];
  const float inv_den = 1.f / (fmaxf(fabsf(qn), expf(-m_new)) + eps);
  if (blockIdx.x == 0 && tid == 0) store_state_scalar(m_out, bh, dtype_state, m_new);

  float vv[VPL];
#pragma unroll
  for (int e = 0; e < VPL; ++e) vv[e] = 0.f;
  if (col_ok) {
    const size_t o = (size_t)bh * DHHV + col;
    if (dtype_qkv == 0) {
#pragma unroll
      for (int e4 = 0; e4 < VPL / 4; ++e4) {
        const f32x4 raw = *(const f32x4*)((const float*)v + o + 4 * e4);
#pragma unroll
        for (int e = 0; e < 4; ++e) vv[4 * e4 + e] = raw[e];
      }
    } else {
#pragma unroll
      for (int e4 = 0; e4 < VPL / 4; ++e4) {
        const uint2 raw = *(const uint2*)((const uint16_t*)v + o + 4 * e4);
        unpack_state2(raw.x, dtype_qkv, vv[4 * e4 + 0], vv[4 * e4 + 1]);   // dtype code 1 bf16, 2 fp16
        unpack_state2(raw.y, dtype_qkv, vv[4 * e4 + 2], vv[4 * e4 + 3]);
      }
    }
  }
  float acc[VPL];
#pragma unroll
  for (int e = 0; e < VPL; ++e) acc[e] = 0.f;
  // C' = f' C + i' k v^T for one piece of row rr; q^T C' accumulates from the fp32 values (before any rounding)
  auto update = [&](const StatePiece<SBF>& cold, int rr) {
    StatePiece<SBF> o;
    const float ikr = ik[rr], qr = qs[rr];
#pragma unroll
    for (int e = 0; e < VPL; ++e) {
      o.x[e] = fa * cold.x[e] + ikr * vv[e];
      acc[e] += qr * o.x[e];
    }
    return o;
  };
  if (col_ok) {
    int r = ty;
    if (have_first) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int rr = r + u * TY;
        store_piece<SBF, MODE>(c_head, c_bytes, (size_t)rr * DHHV + col, update(cfirst[u], rr));
      }
      r += UNROLL * TY;
    }
    for (; r + (UNROLL - 1) * TY < DHQK; r += UNROLL * TY) {
      StatePiece<SBF> c[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) c[u] = load_piece<SBF, NONTEMPORAL>(c_in, cbase + (size_t)(r + u * TY) * DHHV);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int rr = r + u * TY;
        store_piece<SBF, MODE>(c_head, c_bytes, (size_t)rr * DHHV + col, update(c[u], rr));
      }
    }
    for (; r < DHQK; r += TY) {
      const StatePiece<SBF> c = load_piece<SBF, false>(c_in, cbase + (size_t)r * DHHV);
      store_piece<SBF, NONTEMPORAL ? kPlain : MODE>(c_head, c_bytes, (size_t)r * DHHV + col, update(c, r));
    }
  }
#pragma unroll
  for (int e = 0; e < VPL; ++e) red[ty * COLS + VPL * tx + e] = acc[e];
  __syncthreads();
  for (int cidx = tid; cidx < COLS; cidx += NTH) {
    if (col0 + cidx < DHHV) {
      float s = 0.f;
#pragma unroll
      for (int y = 0; y < TY; ++y) s += red[y * COLS + cidx];
      s *= inv_den;
      const size_t o = (size_t)bh * DHHV + col0 + cidx;
      store_state_scalar(h, o, dtype_qkv, s);   // fp32, bf16 or fp16
    }
  }
}

template <int COLS, int TY, int UNROLL, int MODE, int SBF>
static const char* launch_step_t(const void* q, const void* k, const void* v, const void* i, const void* f,
                                 const void* c_in, const void* n_in, const void* m_in, void* h, void* c_out,
                                 void* n_out, void* m_out, int B, int NH, int DHQK, int DHHV, float eps,
                                 int dtype_qkv, int dtype_gates, hipStream_t stream) {
  const size_t smem = (size_t)(2 * DHQK + TY * COLS) * sizeof(float);
  if (smem > 64 * 1024) return "mlstm_hip_step: DHQK too large for the LDS staging";
  dim3 grid((DHHV + COLS - 1) / COLS, B * NH);
  hipLaunchKernelGGL((step_kernel<COLS, TY, UNROLL, MODE, SBF>), grid, dim3((COLS / StatePiece<SBF>::N) * TY), smem,
                     stream, q, k, v, i, f, c_in, n_in, m_in, h, c_out, n_out, m_out, DHQK, DHHV, eps, dtype_qkv,
                     dtype_gates);
  return nullptr;
}

const char* launch_step(const void* q, const void* k, const void* v, const void* i, const void* f,
                        const void* c_in, const void* n_in, const void* m_in, void* h, void* c_out,
                        void* n_out, void* m_out, int B, int NH, int DHQK, int DHHV, float eps,
                        int dtype_qkv, int dtype_gates, int dtype_state, hipStream_t stream) {
  if (B <= 0 || NH <= 0 || DHQK <= 0 || DHHV <= 0) return "mlstm_hip_step: non-positive dimension";
  const bool sbf = dtype_state != 0;
  if (DHHV % (sbf ? 8 : 4) != 0)
    return sbf ? "mlstm_hip_step: DHHV must be a multiple of 8 for a 16-bit state" : "mlstm_hip_step: DHHV must be a multiple of 4";
  if ((long long)B * NH > 65535) return "mlstm_hip_step: B*NH exceeds 65535";
  // Tile shapes from a sweep on MI355X (B = 16/64/256, NH = 8, 256 x 512 fp32 state).  A state larger than the 256 MB
  // memory-side cache streams past the caches with non-temporal accesses: 256-column slices, 8 row groups, 16 rows
  // in flight per lane.  A smaller one is best left cacheable (it is re-read by the next step) and has few
  // workgroups per CU: 128-column slices with 16 row groups, the first 16 rows per lane requested before the
  // prologue.  The crossover was measured between a 268 MB state (cacheable 79 us, streaming 90 us) and a 403 MB
  // state (156 us against 133 us).  A bfloat16 or float16 state uses the same shapes with lanes of eight columns (half as many
  // lanes per row segment), so every lane still moves 16 bytes per access.
  const size_t state_bytes = (size_t)B * NH * DHQK * DHHV * (sbf ? 2 : 4);
  const bool stream_past_cache = state_bytes > ((size_t)320 << 20);
#define MLSTM_STEP_ARGS q, k, v, i, f, c_in, n_in, m_in, h, c_out, n_out, m_out, B, NH, DHQK, DHHV, eps, dtype_qkv, dtype_gates, stream
#define MLSTM_STEP_PICK(COLS_, TY_, UN_, NT_)                                                          \
  {                                                                                                     \
    if (dtype_state == 1) return launch_step_t<COLS_, TY_, UN_, NT_, 1>(MLSTM_STEP_ARGS);               \
    if (dtype_state == 2) return launch_step_t<COLS_, TY_, UN_, NT_, 2>(MLSTM_STEP_ARGS);               \
    return launch_step_t<COLS_, TY_, UN_, NT_, 0>(MLSTM_STEP_ARGS);                                      \
  }
  if (DHHV % 256 == 0 && stream_past_cache) MLSTM_STEP_PICK(256, 8, 16, kNonTemporal)
  if (stream_past_cache) MLSTM_STEP_PICK(128, 8, 8, kNonTemporal)
  // Below it, the first batch is as many rows as every row group has, up to 16: what is left over is read one row after the other.
  // us, 16 rows at a time / so (128/256 heads, inputs and state new to the caches): 16 x 16 heads 13.9 / 13.3, 64 x 16 60.2 / 53.3, 100 x 16
  // 100.5 / 86.3, with 16-bit states 64 x 16 42.5 / 29.7; 64/64, 512 x 4 26.5 / 20.7.
  // Heads of 64 rows and columns: slices of 64, half the lanes of one of 128 have nothing to do (64/64, 4 heads, 128 / 64 columns: B=200
  // 10.5 / 9.1, of which the host takes all, B=400 16.1 / 11.0, B=512 19.8 / 12.5, 16-bit states 14.1 / 9.1).
  // Write-through where many workgroups of up to 64 KB follow one another on a CU, and the memory-side cache holds the old state beside
  // the new one: us, plain / write-through, the state of one call the next one's input: 128/256, 32 x 16 heads (64 MB) 24.4 / 22.9;
  // 64/128, 128 x 8 (32 MB) 17.1 / 15.1, 400 x 8 42.0 / 37.9; 16-bit states, 256/512 32 x 8 (64 MB) 28.9 / 27.6, 128/256 64 x 16 26.7 / 24.2.
  // Where a single round of workgroups fills the chip the stores wait for it: with 32 MB or less (128/256, 16 x 16, in place 10.1 / 12.4),
  // 12 MB where a workgroup has 32 KB (64/128, 32 x 8 5.8 / 6.3), and with slices of 128 KB (256/512, 16 x 8 20.6 / 23.0).  With more than
  // the cache holds it is memory either way (128/256, 64 x 16, other states in between 53.3 / 57.3).  16-bit states of more rows gain as
  // well (512/1024, 40 MB 21.8 / 21.1, 96 MB 41.8 / 40.6).  Slices of 64 columns from 20 MB on (64/64, 16 MB 7.7 / 7.8, 24 MB 11.2 / 10.0; 100/64 8.2 /
  // 8.8, 11.5 / 11.1), 16-bit states from 12 (64/64, 8 MB 6.3 / 6.8, 16 MB 9.4 / 8.8).
  const bool narrow = DHHV <= 64 && DHQK < 128;
  const size_t slice_bytes = (size_t)128 * DHQK * (sbf ? 2 : 4);
  const size_t least = narrow ? (sbf ? 12 : 20) : slice_bytes <= 32768 ? 12 : 32;  // MB
  // (Stores of 16 bytes: at multiples of 16 only.)
  const bool through = (uintptr_t)c_out % 16 == 0 && (sbf || slice_bytes <= 65536) && state_bytes > least << 20 && state_bytes <= (size_t)112 << 20;
#define MLSTM_STEP_ROWS(MODE_)                                       \
  {                                                                  \
    if (narrow) MLSTM_STEP_PICK(64, 16, 4, MODE_)                    \
    if (DHQK >= 128) MLSTM_STEP_PICK(128, 16, 8, MODE_)              \
    MLSTM_STEP_PICK(128, 16, 4, MODE_)                               \
  }
  if (DHQK >= 256) {
    if (through && dtype_state == 1) return launch_step_t<128, 16, 16, kWriteThrough, 1>(MLSTM_STEP_ARGS);
    if (through) return launch_step_t<128, 16, 16, kWriteThrough, 2>(MLSTM_STEP_ARGS);  // (no float32 state)
    MLSTM_STEP_PICK(128, 16, 16, kPlain)
  }
  if (through) MLSTM_STEP_ROWS(kWriteThrough)
  MLSTM_STEP_ROWS(kPlain)
#undef MLSTM_STEP_ROWS
#undef MLSTM_STEP_PICK
#undef MLSTM_STEP_ARGS
}

}  // namespace mlstm
