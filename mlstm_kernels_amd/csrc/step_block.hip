// Recurrent mLSTM over T tokens in one launch, on the matrix cores: the recurrence of step_seq.hip for 16-bit q, k, v,
// tokens taken in blocks of up to 32.
//
// With f'_t, i'_t, m_t the stabilised gates of the step (step.hip), D[t][j] = i'_j f'_{j+1} ... f'_t and b_t = f'_1 ... f'_t
// over the tokens of a block, C and n the state before it:
//   h_t = ( b_t q_t^T C + sum_{j<=t} D[t][j] (q_t . k_j) v_j ) / sqrt(d) / ( max(|the same with n in place of C|, exp(-m_t)) + eps )
//   C'  = b_T C + sum_j k_j (D[T][j] v_j)^T,     n' = b_T n + sum_j D[T][j] k_j
//
// What bounded the token-by-token kernel is vector arithmetic: three operations per state element and token.  As products
// of blocks the same work is a few dozen matrix instructions, and what is left is one pass over the state: measured in
// bf16 with fp32 states against the token-by-token kernel (us): B = 16, NH = 8, 256/512: 2 tokens 37 -> 32, 16 tokens
// 63 -> 35 (3.8 TB/s of state), 32 tokens 89 -> 39, 128 tokens 250 -> 105; B = 1, 16 tokens: 32 -> 10; 16 x 4 heads of
// 512/1024, 16 tokens: 208 -> 62; 64 x 8 heads of 64/128, 128 tokens: 155 -> 50.  Register budgets for three waves a SIMD
// spill: 32 tokens 38 -> 47.
//
// Arithmetic: as exact as the fp32 recurrence.  q, k and v are exact in bf16 (an fp16 value is the exact sum of two bf16
// values); the other operand of every product -- the state, the gated scores, the weighted values, all fp32 -- is split
// into three bf16 parts whose sum carries 24 bits, one matrix instruction each; sums are fp32.  The gate products are
// formed by successive multiplication like in the recurrence, not from differences of prefix sums.
// Values that are not finite, or so large that a product or sum of the block form could overflow where the recurrence does
// not (kHugeRow, kHugeState), do not go through it: zero times them is NaN at the earlier tokens of the block, and the parts
// of a split infinity are an infinity and a NaN.  From such a block on tokens are taken one at a time in the
// recurrence's own fp32 arithmetic (one_by_one), whose results are those of step_seq.hip, infinities and NaN included.
// Looking costs 0.4 us of 32 at 16 x 8 heads of 256/512 and 16 tokens and 2 of 98 at 128 (the waves wait for the state in front
// of the gating instead of behind it; a barrier of its own behind it costs 2 of 32).
//
// Split: a wave owns 64 rows x 64 value columns of the state of one (batch, head), in registers from the first token to
// the last (64 per lane; lane r of a half holds columns 2 r and 2 r + 1, so rows move in 8-byte pieces of whole 256-byte
// runs).  The waves of a workgroup cover all rows of 64 or 128 columns: everything up to the division is linear in the
// rows, so each works on its own rows alone -- read-out, scores, their product with V, q . n -- and the sums over the row
// groups are taken once per block, in LDS, on the way to h.
// The accumulator layout of C (lane r, half hh, entry i: row 8 (i / 4) + 4 hh + i % 4, column r) is, in eights, the operand
// layout of C^T for a contraction over rows, when q is read in the same order: no movement between update and read-out;
// the score block likewise becomes the operand of its product with V where it lies.
#include "common.h"
#include "kernels.h"

namespace mlstm {
namespace {
constexpr int kBlk = 32;     // tokens per block
constexpr int kDS = 36;      // row stride of the table D (floats)
constexpr int kRowS = 100;   // row stride of the 64-entry K and V rows: plain and transposing reads fall on distinct banks
constexpr int kOutS = 68;    // row stride of the partial sums (floats)
// With q, k, v below 2^30 (fp16: finite) and C, n below 2^80 before the first block no sum of their products overflows: a
// token adds less than 2^60 to the state, so that it needs no second look in later blocks, a score of 64 rows stays below
// 2^66 and a block's share of h below 2^128 for any number of tokens that memory can hold.
constexpr uint16_t kHugeRow = 0x4e80;                 // 2^30 in bf16
constexpr float kHugeState = 1.2089258196146292e24f;  // 2^80

// eight fp32 values -> three bf16 fragments whose sum is the value to 24 bits
__device__ __forceinline__ void split3(const float* x, Frag& a, Frag& b, Frag& c) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t h = pack_bf16x2(x[2 * p], x[2 * p + 1]);
    const float r0 = x[2 * p] - __uint_as_float(h << 16), r1 = x[2 * p + 1] - __uint_as_float(h & 0xffff0000u);
    const uint32_t m = pack_bf16x2(r0, r1);
    a.w[p] = h;
    b.w[p] = m;
    c.w[p] = pack_bf16x2(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
  }
}
// acc += A B for A = eight fp32 values per lane, B = 16-bit values (both exact)
template <bool F16>
__device__ __forceinline__ void mfma_exact(f32x16& acc, const float* x, const Frag& in) {
  Frag a, b, c;
  split3(x, a, b, c);
  if constexpr (!F16) {
    mfma32(acc, c, in);
    mfma32(acc, b, in);
    mfma32(acc, a, in);
  } else {
    Frag u, w;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float x0 = lo2<true>(in.w[p]), x1 = hi2<true>(in.w[p]);
      u.w[p] = pack_bf16x2(x0, x1);
      w.w[p] = pack_bf16x2(x0 - __uint_as_float(u.w[p] << 16), x1 - __uint_as_float(u.w[p] & 0xffff0000u));
    }
    mfma32(acc, c, w);
    mfma32(acc, b, w);
    mfma32(acc, c, u);
    mfma32(acc, a, w);
    mfma32(acc, b, u);
    mfma32(acc, a, u);
  }
}
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
// the larger magnitudes, as bit patterns, of two 16-bit values each
__device__ __forceinline__ u16x2 max_magnitude(u16x2 a, uint4 w) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    a = __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, (&w.x)[e] & 0x7fff7fffu));
  return a;
}
__device__ __forceinline__ float lane_value(float x, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); }
}  // namespace

// F16: q, k, v and h are float16 instead of bfloat16; SDT: state type (0 fp32, 1 bf16, 2 fp16); MODE: 1 up to 16
// tokens, 2 up to 32, 3 more (several blocks); THROUGH: the state is written through the caches.  rows: tokens of the largest block
template <bool F16, int SDT, int MODE, bool THROUGH>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void step_block_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, const void* __restrict__ ig,
    const void* __restrict__ fg, const void* c_in, const void* n_in, const void* m_in, uint16_t* __restrict__ h, void* c_out,
    void* n_out, void* m_out, int T, int DHQK, int DHHV, float eps, int dtype_gates, int rows) {
  constexpr bool MULTI = MODE == 3;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int nw = blockDim.x >> 6, RG = DHQK >> 6, CG = nw / RG;
  const int wave_bytes = max(kBlk * kRowS * 2, rows * kOutS * 4);
  float* const Dt = (float*)smem_raw;               // [32][kDS]
  float* const bt = Dt + kBlk * kDS;                // [32] b_t
  float* const et = bt + kBlk;                      // [32] exp(-m_t)
  float* const den = et + kBlk;                     // [nw][32] partial denominators
  float* const nvec = den + nw * kBlk;              // [nw][64] n of the wave's rows
  int* const odd = (int*)(nvec + nw * 64);          // [nw] whether the wave's rows or its state hold a value that is too large
  uint16_t* const Vs = (uint16_t*)(odd + 8);        // [CG][32][kRowS] v rows, even columns first
  unsigned char* const wave_mem = (unsigned char*)(Vs + CG * kBlk * kRowS);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, cg = wave / RG;
  const int r = lane & 31, hh = lane >> 5;
  const BlockId id = xcd_block_id();
  const int bh = id.y;
  const int col = (id.x * CG + cg) * 64, row0 = rg * 64;
  uint16_t* const Ks = (uint16_t*)(wave_mem + wave * wave_bytes);  // [32][kRowS] this wave's 64 entries of the k rows
  float* const Ps = (float*)Ks;                                    // [rows][kOutS] then: this wave's share of the read-out
  float* const nw_v = nvec + wave * 64;
  const float scale = rsqrtf((float)DHQK);

  float m = wave == 0 ? load_state_scalar(m_in, bh, SDT) : 0.f;
  float nreg = load_state_scalar(n_in, (size_t)bh * DHQK + row0 + lane, SDT);
  f32x16 C[2][2];  // [row tile][even, odd columns]
  const size_t c_base = ((size_t)bh * DHQK + row0) * DHHV + col;   // uniform; plus a 32-bit offset per lane
  const uint32_t c_lane = 4 * hh * DHHV + 2 * r;

  // tokens t0 to t0 + nb; false, with nothing done, if they have to be taken one by one (the same in all waves)
  auto block = [&](int t0, int nb, bool first) __attribute__((always_inline)) {
    const size_t tok = (size_t)bh * T + t0;
    // ---- the block's rows (zeros past the last token): k and v through LDS, q straight into operands
    uint4 kraw[4];
    uint4 vraw[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int row = 8 * x + (lane >> 3);
      kraw[x] = *(const uint4*)(k + (tok + min(row, nb - 1)) * DHQK + row0 + 8 * (lane & 7));
      if (row >= nb) kraw[x] = make_uint4(0, 0, 0, 0);
    }
    // 256 pieces of v over the RG waves of the column group
    const int vn = 4 / RG;  // whole rounds (0 for eight row groups: half of the waves take one)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (x < max(vn, 1)) {
        const int row = min(8 * (x * RG + rg) + (lane >> 3), kBlk - 1);
        vraw[x] = *(const uint4*)(v + (tok + min(row, nb - 1)) * DHHV + col + 8 * (lane & 7));
        if (row >= nb) vraw[x] = make_uint4(0, 0, 0, 0);
      }
    }
    Frag Q[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        Q[s].d[half] = *(const uint2*)(q + (tok + min(r, nb - 1)) * DHQK + row0 + 16 * s + 8 * half + 4 * hh);
      }
    float fraw = 0.f, iraw = 0.f;
    if (wave == 0) {
      const size_t o = tok + min(lane, nb - 1);
      fraw = load_scalar(fg, o, dtype_gates);
      iraw = load_scalar(ig, o, dtype_gates);
    }
    if (first) {  // requested behind the rows, so that the tables are made while the state is on its way
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const size_t o = c_base + (size_t)(32 * b + 8 * (i / 4) + (i % 4)) * DHHV;
          float x0, x1;
          if constexpr (SDT == 0) {
            const float2 x = *(const float2*)((const float*)c_in + o + c_lane);
            x0 = x.x, x1 = x.y;
          } else {
            unpack_state2(*(const uint32_t*)((const uint16_t*)c_in + o + c_lane), SDT, x0, x1);
          }
          C[b][0][i] = x0;
          C[b][1][i] = x1;
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!first) __syncthreads();  // the previous block's tables, rows and sums are no longer read
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      uint16_t* const p = Ks + (8 * x + (lane >> 3)) * kRowS + 8 * (lane & 7);
      *(uint2*)p = make_uint2(kraw[x].x, kraw[x].y);
      *(uint2*)(p + 4) = make_uint2(kraw[x].z, kraw[x].w);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int row = 8 * (x * RG + rg) + (lane >> 3);
      if (x < max(vn, 1) && row < kBlk) {
        uint16_t* const p = Vs + (cg * kBlk + row) * kRowS + 4 * (lane & 7);
        const uint4 w = vraw[x];
        *(uint2*)p = make_uint2(__builtin_amdgcn_perm(w.y, w.x, 0x05040100), __builtin_amdgcn_perm(w.w, w.z, 0x05040100));
        *(uint2*)(p + 32) = make_uint2(__builtin_amdgcn_perm(w.y, w.x, 0x07060302), __builtin_amdgcn_perm(w.w, w.z, 0x07060302));
      }
    }
    nw_v[lane] = nreg;
    bool huge;
    {  // (in front of the tables: the barrier behind them waits for the wave that makes them)
      u16x2 big = {0, 0};
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        big = max_magnitude(big, kraw[x]);
        if (x < max(vn, 1)) big = max_magnitude(big, vraw[x]);
      }
      huge = max(big.x, big.y) >= (F16 ? 0x7c00 : kHugeRow);
    }
    float m_next = m;
    // ---- gate tables, by the first wave: lane t holds the gates of token t (past the last token: keep everything, add
    // nothing), then lane j the column j of D
    if (wave == 0) {
      const float lf = log_sigmoid(fraw), ii = iraw;
      float mm = m, m_prev = m, m_new = m;
      for (int t = 0; t < nb; ++t) {
        if (lane == t) m_prev = mm;
        mm = fmaxf(lane_value(lf, t) + mm, lane_value(ii, t));
        if (lane == t) m_new = mm;
      }
      const float fa = lane < nb ? expf(lf + m_prev - m_new) : 1.f;
      const float ia = lane < nb ? expf(ii - m_new) : 0.f;
      if (lane < kBlk) et[lane] = expf(-m_new);
      float x = 0.f, b = 1.f, b_keep = 1.f;
      for (int t = 0; t < nb; ++t) {
        const float ft = lane_value(fa, t);
        b *= ft;
        x = lane == t ? ia : x * ft;
        if (lane == t) b_keep = b;
        if (lane < kBlk) Dt[t * kDS + lane] = x;
      }
      if (lane < kBlk) bt[lane] = b_keep;
      m_next = mm;
    }
    // ---- this wave's part of the scores (rows j, columns t) and of q . n, from its own rows alone.  Everything works on
    // columns t = r; those past the last token hold rubbish and are not stored.
    f32x16 sc;
    float qn = 0.f;
    asm volatile("" ::: "memory");  // (the rows and n were written by this wave)
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      Frag A;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        A.d[half] = *(const uint2*)(Ks + r * kRowS + 16 * ks + 8 * half + 4 * hh);
        const float4 nv = *(const float4*)(nw_v + 16 * ks + 8 * half + 4 * hh);
        const uint2 w = Q[ks].d[half];
        qn += lo2<F16>(w.x) * nv.x + hi2<F16>(w.x) * nv.y + lo2<F16>(w.y) * nv.z + hi2<F16>(w.y) * nv.w;
      }
      mfma32<F16>(sc, A, Q[ks]);
    }
    {  // (q here, where it is needed anyway)
      u16x2 bq = {0, 0};
#pragma unroll
      for (int x = 0; x < 4; ++x) bq = max_magnitude(bq, Q[x].u);
      huge |= max(bq.x, bq.y) >= (F16 ? 0x7c00 : kHugeRow);
    }
    if (first) {  // (behind all that does not need it: the state may still be on its way)
      float top = fabsf(nreg);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          top = __builtin_elementwise_maximum(__builtin_elementwise_maximum(top, fabsf(C[b][0][i])), fabsf(C[b][1][i]));
      huge |= !(top < kHugeState);
    }
    {
      const bool any_huge = __any(huge);
      if (lane == 0) odd[wave] = any_huge;
    }
    __syncthreads();
    if (__builtin_expect(__any(lane < nw && odd[lane < nw ? lane : 0]), 0)) return false;
    m = m_next;
    const float* const Dlast = Dt + (nb - 1) * kDS;
    // ---- the scores gated, the wave's part of the denominators
    float P[16];
    {
      float rsum = 0.f;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const float4 dv = *(const float4*)(Dt + r * kDS + 8 * g4 + 4 * hh);
        const float dd[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          P[4 * g4 + e] = sc[4 * g4 + e] * scale * dd[e];
          rsum += P[4 * g4 + e];
        }
      }
      float dp = __builtin_fmaf(bt[r] * scale, qn, rsum);
      dp += __shfl_xor(dp, 32);
      den[wave * kBlk + r] = dp;
    }
    // ---- read-out: Out^T[w][t] = b_t C^T q / sqrt(d) + V^T P
    f32x16 out[2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < 16; ++i) out[e][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        float x[8];
#pragma unroll
        for (int y = 0; y < 8; ++y) x[y] = C[ks / 2][e][8 * (ks % 2) + y];
        mfma_exact<F16>(out[e], x, Q[ks]);
      }
    {
      const float s = bt[r] * scale;
      out[0] *= s;
      out[1] *= s;
    }
    // ---- state: C = b_T C + K^T (D[T] . V)
    {
      const float bT = bt[nb - 1];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 2; ++e) C[b][e] *= bT;
    }
    const int q16 = (lane >> 4) & 1, i16 = lane & 15;
    const int tr = (4 * hh + (i16 >> 2)) * kRowS + 16 * q16 + 4 * (i16 & 3);
#pragma unroll
    for (int js = 0; js < (MODE == 1 ? 1 : 2); ++js) {
      Frag A[2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int half = 0; half < 2; ++half) A[b].d[half] = lds_read_tr16(Ks + tr + (16 * js + 8 * half) * kRowS + 32 * b);
      const float4 d0 = *(const float4*)(Dlast + 16 * js + 4 * hh), d1 = *(const float4*)(Dlast + 16 * js + 8 + 4 * hh);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        Frag V;
#pragma unroll
        for (int half = 0; half < 2; ++half) V.d[half] = lds_read_tr16(Vs + cg * kBlk * kRowS + tr + (16 * js + 8 * half) * kRowS + 32 * e);
        // out += V^T P: the exact operand is the second one here (the layouts of both are the same)
        {
          Frag a, b, c;
          split3(P + 8 * js, a, b, c);
          if constexpr (!F16) {
            mfma32(out[e], V, c);
            mfma32(out[e], V, b);
            mfma32(out[e], V, a);
          } else {
            Frag u, w;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const float x0 = lo2<true>(V.w[p]), x1 = hi2<true>(V.w[p]);
              u.w[p] = pack_bf16x2(x0, x1);
              w.w[p] = pack_bf16x2(x0 - __uint_as_float(u.w[p] << 16), x1 - __uint_as_float(u.w[p] & 0xffff0000u));
            }
            mfma32(out[e], w, c);
            mfma32(out[e], w, b);
            mfma32(out[e], u, c);
            mfma32(out[e], w, a);
            mfma32(out[e], u, b);
            mfma32(out[e], u, a);
          }
        }
        float x[8] = {lo2<F16>(V.w[0]) * d0.x, hi2<F16>(V.w[0]) * d0.y, lo2<F16>(V.w[1]) * d0.z, hi2<F16>(V.w[1]) * d0.w,
                      lo2<F16>(V.w[2]) * d1.x, hi2<F16>(V.w[2]) * d1.y, lo2<F16>(V.w[3]) * d1.z, hi2<F16>(V.w[3]) * d1.w};
        Frag w1, w2, w3;
        split3(x, w1, w2, w3);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          if constexpr (!F16) {
            mfma32(C[b][e], A[b], w3);
            mfma32(C[b][e], A[b], w2);
            mfma32(C[b][e], A[b], w1);
          } else {
            Frag u, w;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const float x0 = lo2<true>(A[b].w[p]), x1 = hi2<true>(A[b].w[p]);
              u.w[p] = pack_bf16x2(x0, x1);
              w.w[p] = pack_bf16x2(x0 - __uint_as_float(u.w[p] << 16), x1 - __uint_as_float(u.w[p] & 0xffff0000u));
            }
            mfma32(C[b][e], w, w3);
            mfma32(C[b][e], w, w2);
            mfma32(C[b][e], u, w3);
            mfma32(C[b][e], w, w1);
            mfma32(C[b][e], u, w2);
            mfma32(C[b][e], u, w1);
          }
        }
      }
    }
    // ---- n: lane d of the wave's 64
    if (MULTI || !first || (id.x == 0 && cg == 0)) {
      float s = 0.f;
      for (int j = 0; j < nb; ++j) s = __builtin_fmaf(Dlast[j], elem_to_f32<F16>(Ks[j * kRowS + lane]), s);
      nreg = __builtin_fmaf(bt[nb - 1], nreg, s);
    }
    // ---- this wave's share of the read-out over its K rows (no other wave reads them; LDS accesses of a wave stay in order)
    asm volatile("" ::: "memory");
    if (r < nb) {
      float* const p = Ps + r * kOutS + 8 * hh;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        *(float4*)(p + 16 * g4) = make_float4(out[0][4 * g4], out[1][4 * g4], out[0][4 * g4 + 1], out[1][4 * g4 + 1]);
        *(float4*)(p + 16 * g4 + 4) = make_float4(out[0][4 * g4 + 2], out[1][4 * g4 + 2], out[0][4 * g4 + 3], out[1][4 * g4 + 3]);
      }
    }
    return true;
  };
  auto finish = [&](int t0, int nb) __attribute__((always_inline)) {  // h of the block: sum over the row groups, divide
    __syncthreads();
    for (int x = rg * 64 + lane; x < nb * 16; x += RG * 64) {
      const int t = x >> 4, c4 = 4 * (x & 15);
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
      float d = 0.f;
      for (int g = 0; g < RG; ++g) {
        const int w = cg * RG + g;
        const float4 y = *(const float4*)((const float*)(wave_mem + w * wave_bytes) + t * kOutS + c4);
        s.x += y.x, s.y += y.y, s.z += y.z, s.w += y.w;
        d += den[w * kBlk + t];
      }
      const float inv = 1.f / (fmaxf(fabsf(d), et[t]) + eps);
      *(uint2*)(h + ((size_t)bh * T + t0 + t) * DHHV + col + c4) = make_uint2(pack2<F16>(s.x * inv, s.y * inv), pack2<F16>(s.z * inv, s.w * inv));
    }
  };

  // tokens t0 to T one by one, as step_seq.hip computes them: vector arithmetic in fp32 on the state where it lies
  auto one_by_one = [&](int t0) __attribute__((always_inline)) {
    if (wave == 0) et[1] = m;  // (the other waves have not followed it)
    __syncthreads();
    m = et[1];
#pragma unroll 1
    for (int t = t0; t < T; ++t) {
      const size_t tok = (size_t)bh * T + t;
      const float lf = log_sigmoid(load_scalar(fg, tok, dtype_gates)), ii = load_scalar(ig, tok, dtype_gates);
      const float m_new = fmaxf(lf + m, ii);
      const float fa = expf(lf + m - m_new), ia = expf(ii - m_new);
      m = m_new;
      const uint32_t vw = *(const uint32_t*)(v + tok * DHHV + col + 2 * r);
      const float v0 = lo2<F16>(vw), v1 = hi2<F16>(vw);
      const uint16_t* const qt = q + tok * DHQK + row0;
      const uint16_t* const kt = k + tok * DHQK + row0;
      nreg = fa * nreg + ia * elem_to_f32<F16>(kt[lane]);
      const float qn = wave_sum(elem_to_f32<F16>(qt[lane]) * scale * nreg);
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const uint2 kw = *(const uint2*)(kt + 32 * b + 8 * g4 + 4 * hh), qw = *(const uint2*)(qt + 32 * b + 8 * g4 + 4 * hh);
          const float kk[4] = {lo2<F16>(kw.x), hi2<F16>(kw.x), lo2<F16>(kw.y), hi2<F16>(kw.y)};
          const float qq[4] = {lo2<F16>(qw.x), hi2<F16>(qw.x), lo2<F16>(qw.y), hi2<F16>(qw.y)};
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            float c0 = C[b][0][4 * g4 + x] * fa, c1 = C[b][1][4 * g4 + x] * fa;
            c0 = __builtin_fmaf(ia * kk[x], v0, c0);
            c1 = __builtin_fmaf(ia * kk[x], v1, c1);
            a0 = __builtin_fmaf(qq[x] * scale, c0, a0);
            a1 = __builtin_fmaf(qq[x] * scale, c1, a1);
            C[b][0][4 * g4 + x] = c0;
            C[b][1][4 * g4 + x] = c1;
          }
        }
      a0 += __shfl_xor(a0, 32);
      a1 += __shfl_xor(a1, 32);
      __syncthreads();  // the sums of the token before are no longer read
      if (hh == 0) *(float2*)(Ps + 2 * r) = make_float2(a0, a1);
      if (lane == 0) den[wave * kBlk] = qn;
      if (tid == 0) et[0] = expf(-m_new);
      finish(t, 1);
    }
  };

  const int nb0 = min(kBlk, T);
  const bool whole = block(0, nb0, true);
  int t0 = whole ? nb0 : 0;
  if (MULTI && whole) {
    finish(0, nb0);
#pragma unroll 1
    while (t0 < T) {
      const int nb = min(kBlk, T - t0);
      if (!block(t0, nb, false)) break;
      finish(t0, nb);
      t0 += nb;
    }
  }
  if (__builtin_expect(t0 < T, 0)) one_by_one(t0);  // (out of the way of the blocks)
  // ---- state out (C may be updated in place: this wave read its whole part before)
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const size_t o = c_base + (size_t)(32 * b + 8 * (i / 4) + (i % 4)) * DHHV;
      if constexpr (SDT == 0) {
        float* const dst = (float*)c_out + o + c_lane;
        if constexpr (THROUGH) store_write_through((uint64_t*)dst, (uint64_t)__float_as_uint(C[b][1][i]) << 32 | __float_as_uint(C[b][0][i]));
        else *(float2*)dst = make_float2(C[b][0][i], C[b][1][i]);
      } else {
        uint32_t* const dst = (uint32_t*)((uint16_t*)c_out + o + c_lane);
        if constexpr (THROUGH) store_write_through(dst, pack_state2(C[b][0][i], C[b][1][i], SDT));
        else *dst = pack_state2(C[b][0][i], C[b][1][i], SDT);
      }
    }
  if (id.x == 0 && cg == 0) store_state_scalar(n_out, (size_t)bh * DHQK + row0 + lane, SDT, nreg);
  if (id.x == 0 && tid == 0) store_state_scalar(m_out, bh, SDT, m);
  if (!MULTI && whole) finish(0, nb0);
}

template <bool F16, int SDT, int MODE, bool THROUGH>
static const char* launch_step_block_t(const StepBlockArgs& a, hipStream_t stream) {
  const int RG = a.DHQK / 64, CG = a.DHHV % 128 == 0 && RG <= 2 ? 2 : 1, nw = RG * CG;
  const int rows = a.T < kBlk ? a.T : kBlk;
  const int wave_bytes = kBlk * kRowS * 2 > rows * kOutS * 4 ? kBlk * kRowS * 2 : rows * kOutS * 4;
  const size_t smem = (size_t)(kBlk * kDS + 2 * kBlk + nw * (kBlk + 64) + 8) * 4 + (size_t)CG * kBlk * kRowS * 2 + (size_t)nw * wave_bytes;
  static LdsLimit lds;
  if (!lds.allow((const void*)step_block_kernel<F16, SDT, MODE, THROUGH>, smem)) return "step_block: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((step_block_kernel<F16, SDT, MODE, THROUGH>), dim3(a.DHHV / (64 * CG), a.BH), dim3(64 * nw), smem, stream,
                     (const uint16_t*)a.q, (const uint16_t*)a.k, (const uint16_t*)a.v, a.i, a.f, a.c_in, a.n_in, a.m_in,
                     (uint16_t*)a.h, a.c_out, a.n_out, a.m_out, a.T, a.DHQK, a.DHHV, a.eps, a.dtype_gates, rows);
  return nullptr;
}
// All of the state is written at the very end, and what then lies in the L2s goes to memory while the next launch waits for it: a
// state of up to 96 MB, which the memory-side cache holds beside the old one, is written through them instead.  us, plain /
// write-through, other states in between and the state of one call the next one's input: 256/512, 8 heads, 16 tokens B=4 12.5 11.9 /
// 11.3 11.5, B=8 17.4 17.4 / 15.5 15.4, B=16 32.8 31.1 / 29.0 27.1, B=24 (96 MB) 46.9 43.0 / 47.4 39.6, B=32 60.0 61.2 / 62.9 61.3; 64 tokens
// B=16 65.1 59.0 / 62.2 57.1; 16 heads of 128/256, B=32 34.9 33.1 / 33.3 29.2; 64/128, 4 tokens B=64 13.4 12.9 / 11.5 11.2.  It gains nothing
// where the same call is repeated on the same state (16 tokens B=16 34.6 / 34.5).  (Non-temporal stores gain the same, B=16 28.2, but the
// next call then reads from memory: 33.2 instead of 27.1.  At multiples of 8 bytes only: two columns in one atomic store.)
template <bool F16, int SDT, int MODE>
static const char* launch_step_block_w(const StepBlockArgs& a, hipStream_t stream) {
  const bool through = (uintptr_t)a.c_out % 8 == 0 && (size_t)a.BH * a.DHQK * a.DHHV * (SDT == 0 ? 4 : 2) <= ((size_t)96 << 20);
  return through ? launch_step_block_t<F16, SDT, MODE, true>(a, stream) : launch_step_block_t<F16, SDT, MODE, false>(a, stream);
}
template <bool F16, int MODE>
static const char* launch_step_block_s(const StepBlockArgs& a, hipStream_t stream) {
  if (a.dtype_state == 0) return launch_step_block_w<F16, 0, MODE>(a, stream);
  return a.dtype_state == 1 ? launch_step_block_w<F16, 1, MODE>(a, stream) : launch_step_block_w<F16, 2, MODE>(a, stream);
}

// 16-bit q, k, v and head dimensions that fill the waves' 64 x 64 parts, a power of two of them so that the rows of v deal
// evenly; there it was faster at every token count, batch and state type tried (1.1 to 5 times).  Everything else -- fp32
// inputs, whose products would need nine matrix instructions, and odd dimensions -- runs the token-by-token kernel.
bool step_block_supported(int DHQK, int DHHV, int dtype_qkv) {
  return dtype_qkv != 0 && (DHQK == 64 || DHQK == 128 || DHQK == 256 || DHQK == 512) && DHHV % 64 == 0;
}
const char* launch_step_block(const StepBlockArgs& a, hipStream_t stream) {
  if (a.dtype_qkv == 2)
    return a.T <= 16 ? launch_step_block_s<true, 1>(a, stream) : a.T <= kBlk ? launch_step_block_s<true, 2>(a, stream) : launch_step_block_s<true, 3>(a, stream);
  return a.T <= 16 ? launch_step_block_s<false, 1>(a, stream) : a.T <= kBlk ? launch_step_block_s<false, 2>(a, stream) : launch_step_block_s<false, 3>(a, stream);
}

}  // namespace mlstm
