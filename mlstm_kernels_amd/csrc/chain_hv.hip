// Chain kernels: the state recurrence and the output that spans value columns in ONE launch (forward: C and H; backward: dC and dV).
//
//   forward, steps of 64 positions in order:       H_s  = [ csc . (Q_s C) + P_s V_s ] / (max(|den|, floor) + eps),  C <- g C + K_s^T (us . V_s)
//   backward, steps of 64 positions from the end:  dV_s = csc . (K_s dC) + P_s^T dH_s,                              dC <- g dC + Q_s^T (us . dH_s)
//
// (formulas of mlstm_kernels/torch/chunkwise/native/fw.py:88-212 and bw.py:67-198 in the reference, chunks of 64.)
// A workgroup owns one (batch, head) and W value columns and walks the whole sequence; its DHQK x W slice of the fp32 state stays
// in accumulator registers.  Against a state scan followed by a kernel over chunks no state goes to memory for the sake of H / dV
// (those that dQ / dK need still do), and the rows are read once instead of twice: 256 + 512 head dimensions move 2.1 GB per 2^19
// token-heads of a forward without a backward instead of 3.7.
//
//   * Eight waves, two a SIMD (256 registers): wave (g, dq) owns 32 columns and, with W = 128, half of the state's rows; the two
//     partial products of a position then meet in LDS.  A state tile of 32 x 32 is at once the accumulator of the update and, rounded,
//     the operand of the product with the state: its rows are taken in the order in which a lane's registers are eight neighbouring
//     ones (the transposing reads of K trade two groups of four), so that it never passes through LDS.
//   * Rows come straight into LDS, swizzled, one step ahead.  Where two sets of tiles fit (64 and 128 state rows) all of them are
//     requested in the first half of a step; with 256 the output-side rows go to a free tile, the other rows and the value rows, in the
//     second half, where the present ones have been read.  Two barriers a step.
//   * What goes through the memory path in the second half, requests and rows of the output, goes out between the matrix instructions of
//     the update: in front of it the waves stood there, and a step ends when its requests are there, not when its output is written.
//     With that, the two sets and the swizzles below, before / after: a step of 256/256 columns 15.9 / 14.1 thousand cycles; us, 128 heads of
//     256/512, 2048 positions with the last state 276 / 260, dV of 1024 133 / 126; 128/256, 128 heads of 2048, 131 / 126 and 123 / 107.
//   * Scores: 10 live tiles of 16 x 16, two a wave, gated in fp32 and written to LDS as operand fragments; q . n on the way as one more
//     operand (three 16-bit parts of n, exactly).
//   * The value rows are scaled in fp32 and enter the state as a 16-bit head and remainder: the state is rounded every 64 positions
//     for the product with it, and that alone is what it loses.  Errors against 64 bits by norm, times 1e-3, with the scan and the
//     kernels over chunks / here, bf16: 128 heads of 256/512, forget gates around 3, H 2.354 / 2.357, dQ 2.373 / 2.364, dK 2.383 / 2.365, dV
//     2.374 / 2.368, gates around 9 2.680 / 2.376, 2.629 / 2.328, 2.690 / 2.324, 2.739 / 2.384; 256 heads of 128/128, gates around 3, H 2.362 /
//     2.371, dV 2.363 / 2.366.  (Rows right behind a step's boundary take most of H from the rounded state; where a normaliser nearly
//     cancels that weighs more: the 99th percentile of the rows is 2 % higher.)
//   * The state takes its decay in every step.  Left in a factor until that reaches 2^-24, with weights that take it, the registers
//     hold up to 2^24 times the state, which overflows with rows of 2^103 and above; and it gained nothing (us, an earlier form of the
//     kernel, forward, backward, so / with the decay: 128 heads of 256/512, 2048 positions 331 303 / 334 306, 256 heads of 1024,
//     128/256 103 97 / 102 96, 128/128 75 70 / 74 69, 64/128 61 60 / 59 60).
// What bounds it: issue.  A step of 256 / 256 columns is 120 matrix and 807 vector instructions a wave, two waves a SIMD, which
// overlap only where they are interleaved (a matrix instruction hides about six of its wave: the schedules below); matrix pipes 50 %
// busy (128 columns: 26 and 29 %), LDS 29 %, 1 to 2 % of that conflicts (20 and 15 % with swizzles for other groups of lanes); 3.4 TB/s,
// every row read once.  us, forward / backward, scan + H (dV) and this: 256/512, 128 heads of 2048 with the last state 377 / 258, of 1024
// 174 / 131 and 167 / 121, of 512 88 / 70 and 80 / 62; 128/256, 256 heads of 1024 141 / 92 and 122 / 90, 128 of 2048 145 / 123 and 129 /
// 105; 128/128, 256 of 1024 102 / 68 and 88 / 59; 64/128, 256 of 1024 81 / 57 and 69 / 47; 256/256, 256 of 512 99 / 75 and 85 / 69.
#include "common.h"
#include "kernels.h"

namespace mlstm {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kStep = 64;

// 16-byte-unit swizzle of the rows of a tile of RB bytes a row.  LDS has 64 banks and serves a 16-byte read in groups of 16 lanes,
// 0-3 12-15 20-27 and 4-11 16-19 28-31 (and the same of lanes 32-63), a transposing read in groups of 32: 32 rows at one unit (a group
// has 16 distinct ones), 16 rows at two units (rows 0-3 and 12-15 at one, 4-11 at the other: hence 0 2 3 1 by groups of four rows, where
// either set is closed under the XOR that parts the units) and 4 consecutive rows at four neighbouring units fall on distinct slots.
// (In the order 0 1 2 3 two rows of every group of the score operands shared a slot; us, 128 heads of 256/512, 2048 positions with
// the last state 291 / 287, forward and backward of 128/256, 128 heads of 2048, 436 / 431.)
template <int RB>
__device__ __forceinline__ int swz(int row) {
  const int g = (row >> 2) & 3, lo = (g >> 1) | (((g ^ (g >> 1)) & 1) << 1);
  return (RB == 128 ? ((row >> 1) & 1) << 2 : (row & 3) << 2) | lo;
}

typedef __attribute__((address_space(3))) unsigned char lds_byte;
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(lds_byte*)p; }

// Buffer descriptor of the rows of one (batch, head): reads past its end give zeros.
__device__ __forceinline__ u32x4 row_desc(const void* base, uint32_t bytes) {
  const uint64_t p = (uint64_t)(uintptr_t)base;
  return u32x4{(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, bytes, 0x00020000u};
}
// The share of wave `wave` in moving a tile of 64 rows of RB bytes to LDS, 16 bytes per lane and 1 KB per instruction without
// registers in between; the 16-byte units of a row are swizzled by swz.  The instruction's own offset counts in memory and in LDS
// (LDS address = M0 + offset + 16 * lane).  `step`: bytes of memory between two instructions' rows (1024 where the rows are
// dense).  In assembly: behind the builtin the compiler waits for every such load in front of every LDS read.  Whoever reads the
// bytes waits with dma_wait() in front of a barrier.  Rows past the end of the sequence arrive as zeros.
template <int RB>
struct DmaTile {
  static constexpr int NP = RB / 128;          // instructions per wave
  static constexpr int RPP = 1024 / RB;        // rows per instruction: 2, 4 or 8
  static_assert(NP == 1 || NP == 2 || NP == 4, "rows of 128, 256 or 512 bytes");
  static __device__ __forceinline__ uint32_t offset(int wave, int lane, uint32_t stride) {  // of the wave's first instruction
    const int row = wave * (NP * RPP) + lane / (RB / 16), unit = lane % (RB / 16);
    return (uint32_t)row * stride + (uint32_t)((unit ^ swz<RB>(row)) << 4);
  }
  // v: offset() + first row * stride
  static __device__ __forceinline__ void load(const u32x4& desc, uint32_t v, uint32_t stride, uint32_t dst, int wave) {
    const uint32_t m0 = dst + wave * (NP * 1024);
    const uint32_t skip = RPP * stride - 1024;
    // how the swizzle of the wave's later rows differs from that of its first ones
    if constexpr (NP == 4) {  // rows 8 w + 2 i + b
      constexpr uint32_t x1 = 8 << 4, x2 = 2 << 4, x3 = 10 << 4;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\t"
                   "buffer_load_dwordx4 %2, %1, 0 offen lds\n\t"
                   "buffer_load_dwordx4 %3, %1, 0 offen offset:1024 lds\n\t"
                   "buffer_load_dwordx4 %4, %1, 0 offen offset:2048 lds\n\t"
                   "buffer_load_dwordx4 %5, %1, 0 offen offset:3072 lds"
                   : : "s"(m0), "s"(desc), "v"(v), "v"((v ^ x1) + skip), "v"((v ^ x2) + 2 * skip), "v"((v ^ x3) + 3 * skip) : "memory");
    } else if constexpr (NP == 2) {  // rows 8 w + 4 i + b
      constexpr uint32_t x1 = 2 << 4;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\t"
                   "buffer_load_dwordx4 %2, %1, 0 offen lds\n\t"
                   "buffer_load_dwordx4 %3, %1, 0 offen offset:1024 lds"
                   : : "s"(m0), "s"(desc), "v"(v), "v"((v ^ x1) + skip) : "memory");
    } else {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\t"
                   "buffer_load_dwordx4 %2, %1, 0 offen lds" : : "s"(m0), "s"(desc), "v"(v) : "memory");
    }
  }
};
// (the wave's last N vector-memory instructions may still be on their way)
template <int N = 0>
__device__ __forceinline__ void dma_wait() {
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | N);  // vmcnt(N), N < 16
  asm volatile("" : : : "memory");
}
// 64 consecutive fp32 values to LDS, one per lane
__device__ __forceinline__ void dma_vec(const float* base, uint32_t v, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dword %1, %2" : : "s"(dst), "v"(v), "s"(base) : "memory");
}

// P holds six fragments (16 other positions o16, 32 positions n32) of 1 KB: those of its three live 32 x 32 blocks
// (fragment o16 + 2 n32, for either direction)

// Nothing is scheduled across: the LDS reads of the next group of matrix instructions stay in front of the present group's.  Left
// alone the compiler reads an operand right before it is used and waits a trip to LDS for every one.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ Frag tr_frag(const uint16_t* lo, const uint16_t* hi) {
  Frag f;
  f.d[0] = lds_read_tr16(lo);
  f.d[1] = lds_read_tr16(hi);
  return f;
}

}  // namespace

template <int DQ, int W, bool F16>
struct ChainLds {  // bytes
  static constexpr int G = W / 32, DS = 8 / G;
  static constexpr int TQ = kStep * DQ * 2, TV = kStep * W * 2, PB = 6144;
  static constexpr int EX = DS == 2 ? 8 * 4096 : 0;
  // Two sets of tiles where they fit (DQ 64 and 128): everything of the next step is requested at the start of this one.
  static constexpr bool kAhead = 4 * TQ + 2 * TV + PB + EX + 12288 <= 160 * 1024;
  static constexpr int kV = (kAhead ? 4 : 3) * TQ, kP = kV + (kAhead ? 2 : 1) * TV, kEx = kP + PB, kVec = kEx + EX;
  // [2][5][64] weights, [2][5][64] gate vectors as they arrive, [8][64] row sums, [4 or 1][64] q . n, decay, n as [DQ] fp32 and (bfloat16)
  // [3][NP] 16-bit parts
  static constexpr int NP = DQ + 16;  // (32 bytes apart: the three rows of a fragment on distinct banks)
  static constexpr int QN = F16 ? 256 : 64;
  static constexpr int kBytes = kVec + (640 + 640 + 512 + QN + 8 + DQ) * 4 + (F16 ? 0 : 3 * NP * 2);
};

// x = sum of three bfloat16 values, exactly (a float32 has 24 significant bits)
__device__ __forceinline__ void split3(float x, uint16_t* dst, int stride) {
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const uint32_t b = pack_bf16x2(x, x);
    dst[p * stride] = (uint16_t)b;
    x -= __uint_as_float(b << 16);
  }
}

// Element offset of unit u0 + u (u0 known at compile time, a multiple of 4, u < 4) of a row with swizzle sw
template <int RB>
__device__ __forceinline__ int unit_ofs(int u0, int u, int sw) {
  constexpr int M = RB == 128 ? 8 : 16;
  return (u0 / M) * (M * 8) + (((u0 % M + u) ^ sw) << 3);
}

// (see opaque(); where there are registers for the addresses of a step they are kept)
template <bool TIGHT>
__device__ __forceinline__ int lane_of(int lane) { return TIGHT ? opaque(lane) : lane; }

// What a launch makes.  kKeptStates: the forward's kept states and nothing else, for a backward that has them recomputed: the same
// arithmetic in the same order, hence the same bits, which the scan, rounding the scaled value rows once, does not have.  us, the whole
// forward / the scan / this: 128 heads of 256/512, 2048 positions 272 / 139 / 152, 1024 131 / 69 / 70; 256 heads of 1024, 128/256 93 / 51 /
// 53, 64/128 58 / 27 / 25.  (The scan's launch, which then ends at once, 6 us.)
enum Kind { kForward, kBackward, kKeptStates };

template <int DQ, int W, int KIND, bool F16>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void chain_hv_kernel(ChainHvArgs a) {
  constexpr bool IS_DV = KIND == kBackward, ROWS = KIND != kKeptStates;  // ROWS: H or dV is made
  if constexpr (!ROWS) {
    if (__builtin_amdgcn_readfirstlane(*a.g.chained) == 0) return;  // the forward's states came from the scan
  }
  using L = ChainLds<DQ, W, F16>;
  constexpr int G = L::G, DS = L::DS;
  constexpr int NDT = DQ / 32 / DS;         // 32-row state tiles of a wave
  constexpr int NO = DS == 1 ? 2 : 1;       // position tiles of 32 whose output a wave finishes
  constexpr int ND = DQ / 16;
  constexpr bool kTight = DQ == 256 && W == 256;
  static_assert(G * DS == 8 && NDT >= 1 && DS <= 2, "eight waves");
  extern __shared__ __align__(16) unsigned char smem[];
  float* const vec = (float*)(smem + L::kVec);  // [2][5][64]: u (t), w (j), us, csc, aux
  float* const raw = vec + 640;                 // [2][5][64]
  float* const rs = raw + 640;                  // [8][64] row sums of P: two waves a position, four lanes each
  float* const qn = rs + 512;                   // [4][64] shares of q . n (bfloat16: one)
  float* const gdl = qn + L::QN;                // [2] decay of the state in a step
  float* const nv = gdl + 8;                    // [DQ] normaliser state
  uint16_t* const npt = (uint16_t*)(nv + DQ);   // [3][NP] the same as three 16-bit parts (bfloat16)

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int g = wave % G, dq = wave / G;        // column group, group of state rows
  const BlockId blk = xcd_block_id();
  const int bh = blk.y, w_tile = blk.x * W;
  const int S = a.S, NC = a.NC, DHHV = a.DHHV;
  const size_t Sp = (size_t)NC * kChunk;
  const int NS = (S + kStep - 1) / kStep;
  const int n_run = ROWS ? NS : 2 * ((NC - 1) / a.stride * a.stride) + 1;  // steps: up to the last kept state
  const bool do_n = KIND == kForward && a.use_nrow;
  const u32x4 Xn_d = row_desc((IS_DV ? a.K : a.Q) + (size_t)bh * S * DQ, (uint32_t)S * DQ * 2);
  const u32x4 Xo_d = row_desc((IS_DV ? a.Q : a.K) + (size_t)bh * S * DQ, (uint32_t)S * DQ * 2);
  const u32x4 Xw_d = row_desc((IS_DV ? a.dH : a.V) + (size_t)bh * S * DHHV + w_tile, ((uint32_t)S * DHHV - w_tile) * 2);
  const uint32_t q_off = DmaTile<DQ * 2>::offset(wave, lane, DQ * 2);
  const uint32_t w_off = DmaTile<W * 2>::offset(wave, lane, DHHV * 2);
  const uint32_t lds0 = lds_addr(smem);
  // rows past the end of the sequence fall outside
  const auto out_d = __builtin_amdgcn_make_buffer_rsrc(a.Out + (size_t)bh * S * DHHV, 0, (uint32_t)S * DHHV * 2, 0x00020000);

  // ---- state: tile dt holds rows 32 (dq NDT + dt) .. +31 in the order 16 (i / 8) + 8 h + i % 8 (register i), column 32 g + r
  f32x16 acc[NDT];
  const int tg0 = dq * NDT;
  const int kb0 = DS == 2 ? 32 * dq : 0, kb1 = 32 - kb0;
  if (a.init != nullptr) {
    const float* src = a.init + ((size_t)bh * DQ + 32 * tg0 + 8 * h) * DHHV + w_tile + 32 * g + r;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[dt][i] = src[(size_t)(32 * dt + 16 * (i / 8) + i % 8) * DHHV];
  } else {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
  }
  if (tid < DQ) {
    const float x = do_n && a.n_init != nullptr ? a.n_init[(size_t)bh * DQ + tid] : 0.f;
    nv[tid] = x;
    if constexpr (!F16) split3(x, npt + tid, L::NP);
  }
  rs[tid] = 0.f;
  for (int x = tid; x < L::PB / 16; x += 512) ((uint4*)(smem + L::kP))[x] = make_uint4(0, 0, 0, 0);

  // gate vectors of step s, by wave 5 or 6 (which have no scores; in turn): requested ...
  auto gates_load = [&](int s) -> float {
    const int ln = opaque(lane), c = s >> 1;
    const uint32_t o = (uint32_t)s * (kStep * 4) + ln * 4;
    const uint32_t dst = lds0 + L::kVec + 640 * 4 + (s & 1) * 1280;
    dma_vec(a.g.u + bh * Sp, o, dst);
    dma_vec(a.g.w + bh * Sp, o, dst + 256);
    dma_vec(a.g.abar + bh * Sp, o, dst + 512);
    dma_vec(a.g.bbar + bh * Sp, o, dst + 768);
    dma_vec((IS_DV ? (a.use_nrow ? a.nrow : a.g.bbar) : a.g.mcomb) + bh * Sp, o, dst + 1024);
    // lane 0: u of the middle of the chunk, lane 1: what the decay is made of, lane 2: m after the chunk
    const bool single = S - c * kChunk <= kStep;
    const float* p = a.g.u + bh * Sp + (size_t)c * kChunk + 63;
    if (ln == 1) p = single ? a.g.gbar + (size_t)bh * NC + c : (s & 1 ? a.g.graw + (size_t)bh * NC + c : a.g.bbar + bh * Sp + (size_t)c * kChunk + 63);
    if (ln == 2) p = a.g.mstates + (size_t)bh * (NC + 1) + c + 1;
    return *p;
  };
  // ... and what they become: weights relative to the middle of the chunk, whose stabiliser is the combined one of position 63
  auto gates_store = [&](int s, float gs) {
    const int ln = opaque(lane), c = s >> 1, odd = s & 1;
    const bool single = S - c * kChunk <= kStep;
    const bool in = s * kStep + ln < S;
    const float u63 = __shfl(gs, 0), gg = __shfl(gs, 1), gm = __shfl(gs, 2);
    const float* const raw_s = raw + (s & 1) * 320;
    const float gu = raw_s[ln], gw = raw_s[64 + ln], gx = raw_s[256 + ln];
    const float A = odd || single ? raw_s[128 + ln] : expf(u63 - gw);  // weight of k v^T in the state after the step
    const float B = odd ? expf(gu - u63) : raw_s[192 + ln];            // weight of the state before the step
    float* v = vec + (s & 1) * 320 + ln;
    v[0] = gu;
    v[64] = gw;
    if (IS_DV) {
      const float rho = in ? (a.use_nrow ? 1.f / (gx + a.eps) : 1.f) : 0.f;
      v[128] = in ? B * a.qk_scale * rho : 0.f;
      v[192] = A;
      v[256] = rho;
    } else {
      v[128] = in ? A : 0.f;
      v[192] = B * a.qk_scale;
      v[256] = gx;
    }
    if (ln == 0) gdl[s & 1] = odd ? expf(gg - u63 - gm) : gg;
  };

  const int s_first = IS_DV ? NS - 1 : 0, s_inc = IS_DV ? -1 : 1;
  uint32_t o_n = 0, o_o = L::TQ, o_f = 2 * L::TQ;  // LDS offsets of the tiles: output-side rows, other rows, free
  auto load_n = [&](int s, uint32_t o) { DmaTile<DQ * 2>::load(Xn_d, q_off + (uint32_t)s * (kStep * DQ * 2), DQ * 2, lds0 + o, wave); };
  auto load_o = [&](int s, uint32_t o) { DmaTile<DQ * 2>::load(Xo_d, q_off + (uint32_t)s * (kStep * DQ * 2), DQ * 2, lds0 + o, wave); };
  uint32_t o_w = L::kV;                            // ... and value rows
  auto load_w = [&](int s, uint32_t o) { DmaTile<W * 2>::load(Xw_d, w_off + (uint32_t)s * (kStep * 2) * (uint32_t)DHHV, DHHV * 2, lds0 + o, wave); };
  if constexpr (ROWS) load_n(s_first, o_n);
  load_o(s_first, o_o);
  load_w(s_first, o_w);
  float gs = 0.f;
  if (wave == 5 + (s_first & 1)) {
    gs = gates_load(s_first);
    dma_wait<>();
    gates_store(s_first, gs);
  }
  if (wave == 6 - (s_first & 1) && n_run > 1) gs = gates_load(s_first + s_inc);
  dma_wait<>();

  // score tiles (16 x 16) of a wave: position block n16 and two neighbouring blocks of the other index, from ob on (mirrored for dV)
  // wave            0  1  2  3  4  5  6  7
  // n16             3  3  2  1  0  -  -  2
  // first / count   0/2 2/2 0/2 0/2 0/1     2/1
  const int sc_n = IS_DV ? 3 - ((0x20001233 >> (4 * wave)) & 3) : ((0x20001233 >> (4 * wave)) & 3);
  const int sc_o = (0x20000020 >> (4 * wave)) & 3;
  const int sc_cnt = (0x10012222 >> (4 * wave)) & 3;
  const int l16 = lane & 15, q4 = lane >> 4;
  const float log2_qk = __log2f(a.qk_scale);
  const size_t NCS = (size_t)(NC + a.stride - 1) / a.stride;

  for (int it = 0; it < n_run; ++it) {
    const int s = s_first + it * s_inc, t0 = s * kStep;
    const int c = s >> 1;
    const bool more = it + 1 < n_run;
    const float* const v = vec + (s & 1) * 320;
    __syncthreads();  // ---- the tiles and vectors of this step are in LDS, the free tile is nobody's
    if (more) {
      if constexpr (L::kAhead) {
        if constexpr (ROWS) load_n(s + s_inc, it & 1 ? 0 : 2 * L::TQ);
      } else {
        if constexpr (ROWS) load_n(s + s_inc, o_f);
        else load_o(s + s_inc, o_f);
      }
    }
    const uint16_t* const Xn = (const uint16_t*)(smem + o_n);
    const uint16_t* const Xo = (const uint16_t*)(smem + o_o);

    if (wave == 6 - (s & 1)) {
      if (more) gates_store(s + s_inc, gs);
    } else if (wave == 5 + (s & 1)) {
      if (it + 2 < n_run) gs = gates_load(s + 2 * s_inc);
    }
    // ---- scores: P (other index, position), gated, rounded, to LDS as operand fragments
    auto scores = [&]() __attribute__((always_inline)) {
    if (sc_cnt > 0) {
      const int ln = lane_of<kTight>(lane);
      const int m16 = ln & 15, qq = ln >> 4;
      const int o16a = IS_DV ? 3 - sc_o : sc_o, o16b = IS_DV ? 2 - sc_o : sc_o + 1;
      const int sw = swz<DQ * 2>(m16);
      const uint16_t* pn = Xn + (16 * sc_n + m16) * DQ;
      const uint16_t* pa = Xo + (16 * o16a + m16) * DQ;
      const uint16_t* pb = Xo + (16 * (o16b & 3) + m16) * DQ;
      const int n = 16 * sc_n + m16;
      const float un = v[(IS_DV ? 64 : 0) + n];
      const float* const ov = v + (IS_DV ? 0 : 64) + 4 * qq;
      const float4 xo[2] = {*(const float4*)(ov + 16 * o16a), *(const float4*)(ov + 16 * (o16b & 3))};
      float4 ro[2];
      if (IS_DV) {
        ro[0] = *(const float4*)(v + 256 + 4 * qq + 16 * o16a);
        ro[1] = *(const float4*)(v + 256 + 4 * qq + 16 * (o16b & 3));
      }
      // q . n on the way: the three parts of n are three rows of one more operand (the other rows of the result are not used)
      constexpr bool kQn = !IS_DV && !F16;
      const uint16_t* pq = npt + (m16 < 3 ? m16 * L::NP : 0) + 8 * qq;
      f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f}, sq = {0.f, 0.f, 0.f, 0.f};
      constexpr int NK = DQ / 32, kDeep = 3;  // operands are read kDeep - 1 steps of 32 head dimensions ahead
      Frag f[kDeep][4];
      auto fetch = [&](int k) {
        const int o = unit_ofs<DQ * 2>(4 * k, qq, sw);
        f[k % kDeep][0].u = *(const uint4*)(pn + o);
        f[k % kDeep][1].u = *(const uint4*)(pa + o);
        f[k % kDeep][2].u = *(const uint4*)(pb + o);
        if (kQn) f[k % kDeep][3].u = *(const uint4*)(pq + 32 * k);
      };
#pragma unroll
      for (int k = 0; k < kDeep - 1; ++k)
        if (k < NK) fetch(k);
      fence();
      float fac[2][4];  // gate factors, while the operands arrive
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const float xov[4] = {xo[x].x, xo[x].y, xo[x].z, xo[x].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ex = IS_DV ? xov[i] - un : un - xov[i];
          fac[x][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(ex, kLog2e, log2_qk));
          if (IS_DV) fac[x][i] *= i == 0 ? ro[x].x : i == 1 ? ro[x].y : i == 2 ? ro[x].z : ro[x].w;
        }
      }
      fence();
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        if (k + kDeep - 1 < NK) fetch(k + kDeep - 1);
        fence();
        mfma16<F16>(sa, f[k % kDeep][1], f[k % kDeep][0]);
        mfma16<F16>(sb, f[k % kDeep][2], f[k % kDeep][0]);
        if (kQn) mfma16<F16>(sq, f[k % kDeep][3], f[k % kDeep][0]);
        fence();
      }
      float rsum = 0.f;
      uint16_t* const pw = (uint16_t*)(smem + L::kP) + (2 * (sc_n >> 1) * 64 + (qq >> 1) * 32 + 16 * (sc_n & 1) + m16) * 8 + (qq & 1) * 4;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int o16 = x == 0 ? o16a : o16b;
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int o = 16 * o16 + 4 * qq + i;
          p[i] = (IS_DV ? n <= o : o <= n) ? (x == 0 ? sa : sb)[i] * fac[x][i] : 0.f;
        }
        if (x == 0 || sc_cnt == 2) {
          rsum += (p[0] + p[1]) + (p[2] + p[3]);
          *(uint2*)(pw + o16 * 512) = make_uint2(pack2<F16>(p[0], p[1]), pack2<F16>(p[2], p[3]));
        }
      }
      if (!IS_DV) rs[(4 * (sc_o >> 1) + qq) * 64 + n] = rsum;
      if (kQn && qq == 0) qn[n] = sq[0] + sq[1] + sq[2];
    }

    // ---- q . n in float32, a quarter of the head dimension by each of the waves with few or no scores (lane = position; the parts
    // of n would be denormal float16 values)
    if (KIND == kForward && F16 && wave >= 4) {
      const int ln = lane_of<kTight>(lane);
      const float* nw = nv + (wave - 4) * (DQ / 4);
      const uint16_t* qr = Xn + ln * DQ;
      float dot[2] = {0.f, 0.f};
      uint4 x[2][2];
      float4 n0[2][2], n1[2][2];
      auto fetch = [&](int k2) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int k = 2 * k2 + e;
          x[k2 & 1][e] = *(const uint4*)(qr + ((((wave - 4) * (DQ / 32) + k) ^ swz<DQ * 2>(ln)) << 3));
          n0[k2 & 1][e] = *(const float4*)(nw + 8 * k);
          n1[k2 & 1][e] = *(const float4*)(nw + 8 * k + 4);
        }
      };
      fetch(0);
#pragma unroll
      for (int k2 = 0; k2 < DQ / 64; ++k2) {
        if (k2 + 1 < DQ / 64) fetch(k2 + 1);
        fence();
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const uint4 w = x[k2 & 1][e];
          const float4 m0 = n0[k2 & 1][e], m1 = n1[k2 & 1][e];
          dot[e] += lo2<F16>(w.x) * m0.x + hi2<F16>(w.x) * m0.y + lo2<F16>(w.y) * m0.z + hi2<F16>(w.y) * m0.w;
          dot[e] += lo2<F16>(w.z) * m1.x + hi2<F16>(w.z) * m1.y + lo2<F16>(w.w) * m1.z + hi2<F16>(w.w) * m1.w;
        }
        fence();
      }
      qn[(wave - 4) * 64 + ln] = dot[0] + dot[1];
    }
    };

    // ---- product with the state: out[k] = position tile (DS == 1: k, else the wave's own one first)
    f32x16 out[2];
    auto product = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) out[k][i] = 0.f;
      {
        const int ln = lane_of<kTight>(lane);
        const int rr = ln & 31, hh = ln >> 5;
        // a wave's rows start at unit 4 tg0: an even number of 16-unit blocks, or (few head dimensions) an XOR on the unit
        constexpr int UB = DQ * 2 == 128 ? 8 : 16;
        const int u0 = 4 * tg0;
        const uint16_t* x0 = Xn + (32 * (DS == 1 ? 0 : dq) + rr) * DQ + (u0 / UB) * (UB * 8);
        const uint16_t* x1 = Xn + (32 * (DS == 1 ? 1 : 1 - dq) + rr) * DQ + (u0 / UB) * (UB * 8);
        const int sw = swz<DQ * 2>(rr) ^ (u0 % UB);
        Frag f[2][2][2];
        auto fetch = [&](int dt) {
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            const int o = unit_ofs<DQ * 2>(4 * dt, 2 * hf + hh, sw);
            f[dt & 1][hf][0].u = *(const uint4*)(x0 + o);
            f[dt & 1][hf][1].u = *(const uint4*)(x1 + o);
          }
        };
        Frag A[2];
        auto round = [&](int i) {
#pragma unroll
          for (int p = 0; p < 4; ++p) A[i & 1].w[p] = pack2<F16>(acc[i >> 1][8 * (i & 1) + 2 * p], acc[i >> 1][8 * (i & 1) + 2 * p + 1]);
        };
        fetch(0);
        round(0);
        fence();
#pragma unroll
        for (int i = 0; i < 2 * NDT; ++i) {
          if (i % 2 == 0 && i / 2 + 1 < NDT) fetch(i / 2 + 1);
          mfma32<F16>(out[0], A[i & 1], f[(i >> 1) & 1][i & 1][0]);
          mfma32<F16>(out[1], A[i & 1], f[(i >> 1) & 1][i & 1][1]);
          if (i + 1 < 2 * NDT) round(i + 1);
        }
#pragma unroll
        for (int i = 0; i < 4 * NDT; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        fence();
      }
      if constexpr (DS == 2) {  // the other half of the sum over the head dimension belongs to the partner wave
        float4* ex = (float4*)(smem + L::kEx + wave * 4096) + lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) ex[64 * k] = make_float4(out[1][4 * k], out[1][4 * k + 1], out[1][4 * k + 2], out[1][4 * k + 3]);
      }
    };
    if constexpr (ROWS) scores();
    if (L::kAhead && more) {
      load_o(s + s_inc, (it & 1 ? 0 : 2 * L::TQ) + L::TQ);
      load_w(s + s_inc, it & 1 ? L::kV : L::kV + L::TV);
    }
    if constexpr (ROWS) product();
    // ---- value rows: transposed fragments, lane = column 32 g + r, eight positions (DS == 2: those of the own position tile first)
    Frag vf[4];
    {
      const int ln = lane_of<kTight>(lane);
      const int i16 = ln & 15, kr = i16 >> 2;
      const int unit = 4 * g + 2 * ((ln >> 4) & 1) + ((i16 & 3) >> 1), sub = 4 * (i16 & 1), row = 8 * (ln >> 5) + kr;
      const uint16_t* base = (const uint16_t*)(smem + o_w) + row * W + sub;
      const uint16_t* lo = base + ((unit ^ swz<W * 2>(row)) << 3);
      const uint16_t* hi = base + 4 * W + ((unit ^ swz<W * 2>(row + 4)) << 3);
#pragma unroll
      for (int j = 0; j < 4; ++j) vf[j] = tr_frag(lo + (j < 2 ? kb0 : kb1) * W + (j & 1) * 16 * W, hi + (j < 2 ? kb0 : kb1) * W + (j & 1) * 16 * W);
    }
    // ---- kept state: before every stride-th chunk (forward), after the last chunk of every group (dV)
    if (a.states != nullptr) {
      const bool chunk_start = IS_DV ? (s & 1) != 0 || s == NS - 1 : (s & 1) == 0;
      const bool keep = chunk_start && (IS_DV ? c == NC - 1 || (c + 1) % a.stride == 0 : c % a.stride == 0);
      if (keep && !(it == 0 && a.skip_zero)) {
        u32x4* dst = (u32x4*)a.states + (((size_t)bh * NCS + c / a.stride) * (size_t)(DHHV / 32) + (w_tile >> 5) + g) * ND * 64 +
                     (size_t)tg0 * 128 + lane;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            uint32_t w[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              float e0 = acc[dt][8 * hf + 2 * p], e1 = acc[dt][8 * hf + 2 * p + 1];
              asm("" : "+v"(e0), "+v"(e1));  // rounded once more: kept from the product they cost its registers (a quarter of the time)
              w[p] = pack2<F16>(e0, e1);
            }
            // rows 8 h + e -> rows 8 (e / 4) + 4 h + e % 4: the halves of the wave trade the middle groups of four
            const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
            const u32x4 f = {x[0], y[0], x[1], y[1]};
            __builtin_nontemporal_store(f, dst + (2 * dt + hf) * 64);
          }
      }
    }
    __syncthreads();  // ---- scores, partial sums; the output-side rows and the value rows have been read
    u32x4 orow[2 * NO];
    if constexpr (ROWS) {
      float4 ex[4];
      if constexpr (DS == 2) {
        const float4* src = (const float4*)(smem + L::kEx + (wave ^ G) * 4096) + lane_of<kTight>(lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) ex[k] = src[64 * k];
      }
      // denominators (lane = position)
      float cs = v[192 + lane], ivl = 1.f;
      {
        const float mc = IS_DV ? 0.f : v[256 + lane];
        float d[12];
        if (!IS_DV) {
#pragma unroll
          for (int x = 0; x < 8; ++x) d[x] = rs[64 * x + lane];
#pragma unroll
          for (int x = 0; x < (F16 ? 4 : 1); ++x) d[8 + x] = qn[64 * x + lane];
        }
        if (!IS_DV) {
          float nmax = 1.f;
          if (do_n) {
            const float q = F16 ? (d[8] + d[9]) + (d[10] + d[11]) : d[8];
            const float sum = cs * q + (((d[0] + d[1]) + (d[2] + d[3])) + ((d[4] + d[5]) + (d[6] + d[7])));
            nmax = fmaxf(fabsf(sum), a.sig_gate ? 1.f : __expf(-mc));
            ivl = 1.f / (nmax + a.eps);
          }
          if (blk.x == 0 && wave == 7) {
            a.nrow_out[bh * Sp + t0 + lane] = nmax;
            // the second half of the last chunk, if no step covers it
            if (s == NS - 1 && (s & 1) == 0) a.nrow_out[bh * Sp + t0 + kStep + lane] = 1.f;
            if (t0 + lane < S) {
              if (a.n_out != nullptr) a.n_out[(size_t)bh * S + t0 + lane] = nmax;
              if (a.m_out != nullptr) a.m_out[(size_t)bh * S + t0 + lane] = mc;
            }
          }
        }
      }
      // from lane = position to lane = position of the wave's tiles, in both halves of the wave
      float csk[NO], iv[NO];
      {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(cs), __float_as_uint(cs), false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(ivl), __float_as_uint(ivl), false, false);
#pragma unroll
        for (int k = 0; k < NO; ++k) {
          csk[k] = __uint_as_float(DS == 1 ? x[k] : (dq ? x[1] : x[0]));
          iv[k] = __uint_as_float(DS == 1 ? y[k] : (dq ? y[1] : y[0]));
        }
      }
      if constexpr (DS == 2) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          out[0][4 * k] += ex[k].x; out[0][4 * k + 1] += ex[k].y; out[0][4 * k + 2] += ex[k].z; out[0][4 * k + 3] += ex[k].w;
        }
      }
#pragma unroll
      for (int k = 0; k < NO; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) out[k][i] *= csk[k];
      // ---- product inside the step
      {
        const uint4* pf = (const uint4*)(smem + L::kP) + lane_of<kTight>(lane);
        if constexpr (DS == 1) {
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
              if (IS_DV ? ks < 2 * k : ks >= 2 * (k + 1)) continue;
              Frag b;
              b.u = pf[(ks + 2 * k) * 64];
              mfma32<F16>(out[k], vf[ks], b);
            }
        } else {
#pragma unroll
          for (int x = 0; x < 2; ++x)  // the diagonal block, then the other one where there is one
            if (x == 0 || dq == (IS_DV ? 0 : 1))
#pragma unroll
              for (int y = 0; y < 2; ++y) {
                Frag b;
                b.u = pf[(2 * (x ^ dq) + y + 2 * dq) * 64];
                mfma32<F16>(out[0], vf[2 * x + y], b);
              }
        }
      }
      // ---- output rows: lane (h, r) holds columns 8 x + 4 h + 0 .. 3 of position r; first the halves of the wave trade, so that it
      // holds eight neighbouring ones, then its rows of 16 lanes, so that four lanes hold the 32 columns of a position
#pragma unroll
      for (int k = 0; k < NO; ++k) {
        uint32_t w[8], o[2][4];
#pragma unroll
        for (int x = 0; x < 8; ++x) w[x] = pack2<F16>(out[k][2 * x] * iv[k], out[k][2 * x + 1] * iv[k]);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const auto p = __builtin_amdgcn_permlane32_swap(w[4 * x], w[4 * x + 2], false, false);
          const auto q = __builtin_amdgcn_permlane32_swap(w[4 * x + 1], w[4 * x + 3], false, false);
          o[x][0] = p[0]; o[x][1] = q[0]; o[x][2] = p[1]; o[x][3] = q[1];
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const auto p = __builtin_amdgcn_permlane16_swap(o[0][x], o[1][x], false, false);
          o[0][x] = p[0]; o[1][x] = p[1];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) orow[2 * k + x] = u32x4{o[x][0], o[x][1], o[x][2], o[x][3]};
      }
    }
    // what goes out during the update (it is what the memory path takes a while for: in front of it the waves stood there)
    auto memory = [&](int i) {
      if constexpr (!L::kAhead) {
        if (i == 0 && ROWS && more) load_o(s + s_inc, o_n);
        if (i == 1 && more) load_w(s + s_inc, o_w);
        i -= 2;
      }
      if constexpr (ROWS) {
        if (i >= 0 && i < 2 * NO) {
          const int n = 32 * (DS == 1 ? i >> 1 : dq) + 16 * (i & 1) + (lane & 15);
          __builtin_amdgcn_raw_buffer_store_b128(orow[i], out_d, (uint32_t)(t0 + n) * (uint32_t)(DHHV * 2) + (uint32_t)(w_tile + 32 * g + 8 * h + (lane & 16)) * 2, 0, 0);
        }
      }
    };
    const float gdec = gdl[s & 1];
    // ---- state update, the scaled value rows as a 16-bit head and remainder; wave w takes rows 32 w .. of the normaliser state
    {
      constexpr bool N = KIND == kForward;  // (nothing reads n behind the other two)
      const int ln = lane_of<kTight>(lane);
      const int i16 = ln & 15, kr = i16 >> 2;
      const int gp = ((i16 & 1) << 1) | ((i16 >> 1) & 1);  // the two middle groups of four rows trade places
      const int row = 8 * (ln >> 5) + kr;
      const int unit = 2 * ((ln >> 4) & 1) + (gp >> 1), sub = 4 * (gp & 1);
      constexpr int UB = DQ * 2 == 128 ? 8 : 16;
      const int ub = 4 * tg0;
      const uint16_t* base = Xo + row * DQ + (ub / UB) * (UB * 8) + sub;
      const int sw_lo = swz<DQ * 2>(row) ^ (ub % UB), sw_hi = swz<DQ * 2>(row + 4) ^ (ub % UB);
      const float* us = v + 128 + 8 * (ln >> 5);
      const int ntile = wave % (DQ / 32);
      const int nunit = 4 * ntile + 2 * ((ln >> 4) & 1) + ((i16 & 3) >> 1), nsub = 4 * (i16 & 1);
      const uint16_t* nbase = Xo + row * DQ + nsub;
      const uint16_t* nlo = nbase + ((nunit ^ swz<DQ * 2>(row)) << 3);
      const uint16_t* nhi = nbase + 4 * DQ + ((nunit ^ swz<DQ * 2>(row + 4)) << 3);
      float nsum = 0.f;
      // Operands are read kAhead state tiles ahead; the scaled value rows of the next 16 positions are made, a quarter at a time,
      // between the matrix instructions of these.
      constexpr int NT = 4 * NDT, kAhead = 3;
      constexpr int kReads = 2 + ((N ? 4 : 2) + NDT - 1) / NDT;
      constexpr int kValu = ((N ? 56 : 40) + 2 * NDT - 1) / (2 * NDT);
      Frag A[4], xn, vh[2], vl[2];
      float4 u0, u1;
      auto row0 = [&](int j) { return (j < 2 ? kb0 : kb1) + 16 * (j & 1); };
      auto fetch = [&](int i) {
        const int j = i / NDT, d = i % NDT;
        A[i & 3] = tr_frag(base + row0(j) * DQ + unit_ofs<DQ * 2>(4 * d, unit, sw_lo), base + (row0(j) + 4) * DQ + unit_ofs<DQ * 2>(4 * d, unit, sw_hi));
      };
      auto weights = [&](int j) {
        u0 = *(const float4*)(us + row0(j));
        u1 = *(const float4*)(us + row0(j) + 4);
        if (N) xn = tr_frag(nlo + row0(j) * DQ, nhi + row0(j) * DQ);
      };
      auto scale = [&](int j, int p) {
        const float x = p == 0 ? u0.x : p == 1 ? u0.z : p == 2 ? u1.x : u1.z, y = p == 0 ? u0.y : p == 1 ? u0.w : p == 2 ? u1.y : u1.w;
        float e0 = lo2<F16>(vf[j].w[p]) * x, e1 = hi2<F16>(vf[j].w[p]) * y;
        // (head and remainder of the same fp32 product: to float16 it may be converted and multiplied in one step)
        if constexpr (F16) asm("" : "+v"(e0), "+v"(e1));
        vh[j & 1].w[p] = pack2<F16>(e0, e1);
        vl[j & 1].w[p] = pack2<F16>(e0 - lo2<F16>(vh[j & 1].w[p]), e1 - hi2<F16>(vh[j & 1].w[p]));
        if (N) {
          nsum = __builtin_fmaf(lo2<F16>(xn.w[p]), x, nsum);
          nsum = __builtin_fmaf(hi2<F16>(xn.w[p]), y, nsum);
        }
      };
      weights(0);
#pragma unroll
      for (int i = 0; i < kAhead; ++i) fetch(i);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] *= gdec;
#pragma unroll
      for (int p = 0; p < 4; ++p) scale(0, p);
      weights(1);
      fence();
      constexpr int NM = L::kAhead ? 2 * NO : 2 * NO + 2;          // memory instructions (or groups of them) to go out
      constexpr int kSeg = NT >= 4 * NM ? NT / 8 : (NT >= NM ? NT / NM : 1);  // state tiles between two of them
#pragma unroll
      for (int i0 = 0; i0 < NT; i0 += kSeg) {
        memory(i0 / kSeg);
        fence();
#pragma unroll
        for (int i = i0; i < i0 + kSeg; ++i) {
          const int j = i / NDT, d = i % NDT;
          if (i + kAhead < NT) fetch(i + kAhead);
          mfma32<F16>(acc[d], A[i & 3], vh[j & 1]);
          mfma32<F16>(acc[d], A[i & 3], vl[j & 1]);
          if (j < 3) {
#pragma unroll
            for (int p = 4 * d / NDT; p < 4 * (d + 1) / NDT; ++p) scale(j + 1, p);
          }
          if (d == NDT - 1 && j < 2) weights(j + 2);
        }
        // a matrix instruction hides about six others of its wave
#pragma unroll
        for (int i = i0; i < i0 + kSeg; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
        }
        fence();
      }
      if (N) {
        nsum += __shfl_xor(nsum, 32);
        const int d = 32 * ntile + (ln & 31);
        const float nn = gdec * nv[d] + nsum;
        if (wave < DQ / 32 && ln < 32) {
          nv[d] = nn;
          if (!F16) split3(nn, npt + d, L::NP);
        }
      }
    }
    // (the rows of the next step were requested before the rows of this one went out)
    dma_wait<ROWS ? 2 * NO : 0>();
    asm volatile("" : "+v"(gs));  // has arrived with them; where it is used the compiler would wait for the rows requested by then
    if constexpr (L::kAhead) {
      o_n = it & 1 ? 0 : 2 * L::TQ;
      o_o = o_n + L::TQ;
      o_w = it & 1 ? L::kV : L::kV + L::TV;
    } else {
      const uint32_t x = o_o;
      o_o = ROWS ? o_n : o_f;
      o_n = o_f;
      o_f = x;
    }
  }

  __syncthreads();
  if (a.final_out != nullptr) {
    float* dst = a.final_out + ((size_t)bh * DQ + 32 * tg0 + 8 * h) * DHHV + w_tile + 32 * g + r;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) dst[(size_t)(32 * dt + 16 * (i / 8) + i % 8) * DHHV] = acc[dt][i];
  }
  if (do_n && a.n_final != nullptr && blk.x == 0) {
    for (int d = tid; d < DQ; d += 512) a.n_final[(size_t)bh * DQ + d] = nv[d];
  }
}

namespace {
template <int DQ, int W, int KIND, bool F16>
const char* launch_t(const ChainHvArgs& a, int BH, hipStream_t stream) {
  static LdsLimit lds;
  constexpr int smem = ChainLds<DQ, W, F16>::kBytes;
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  if (!lds.allow((const void*)chain_hv_kernel<DQ, W, KIND, F16>, smem)) return "chain_hv: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((chain_hv_kernel<DQ, W, KIND, F16>), dim3(a.DHHV / W, BH), dim3(512), smem, stream, a);
  return nullptr;
}
template <int DQ, int W, int KIND>
const char* launch_f(const ChainHvArgs& a, int BH, hipStream_t stream) {
  return a.f16 ? launch_t<DQ, W, KIND, true>(a, BH, stream) : launch_t<DQ, W, KIND, false>(a, BH, stream);
}
template <int DQ, int W>
const char* launch_w(const ChainHvArgs& a, int BH, int kind, hipStream_t stream) {
  if (kind == kBackward) return launch_f<DQ, W, kBackward>(a, BH, stream);
  return kind == kForward ? launch_f<DQ, W, kForward>(a, BH, stream) : launch_f<DQ, W, kKeptStates>(a, BH, stream);
}
// Value columns of a workgroup, 0: another kernel is the better one.
//  * One workgroup takes a CU and the launch as long as its rounds: the last one has to be nearly full.  256 columns are the more
//    efficient form; with 128 the state's rows are shared by two waves that both scale the value rows, and what is gained is less.  The
//    lines, 85 and 95 %, lie between 96 and 128 heads of 256/512 (192 and 256 workgroups of 256) and between 112 and 128 of 128/256 (of
//    128), where an earlier form of this kernel crossed scan + H.  The present one is past it at 75 and 87 % (scan + H / so: 96 heads of
//    1024 135 / 112, dV 129 / 104, 128 175 / 131; 128/256, 112 heads of 2048 136 / 115, dV 122 / 99): they could lie lower.  Not for half
//    of the heads of 256/512, which would be faster (64 heads, scan + stream_hv / so: forward with the last state, 512 positions 63 / 49,
//    1000 107 / 89, 2000 201 / 169; forward and backward, 512 151 / 155, 1000 292 / 294, 2048 599 / 574): H is a little further from 64
//    bits than theirs (errors times 1e-3, gates around 3, 6, 9: 1000 positions 2.357 2.343 2.353 / 2.365 2.372 2.367, 2000 2.355 2.411
//    2.365 / 2.363 2.379 2.375), and where only a forward without a gradient gains it would not have the bits of one with a gradient.
//  * Rows move to LDS in pieces of 16 bytes without registers in between, and rows of the output leave through a buffer descriptor, 16
//    bytes a lane: both ask for addresses that are multiples of 16; the other kernels read and write theirs with ordinary instructions,
//    which do not.
//  * Up to 256 positions the other kernels need no state at all and are faster (256/512, 512 heads of 256: forward 117 / 136, backward
//    87 / 126); at 320 128 heads take 75 / 47 and 65 / 43.
//  * Longer sequences and several rounds are no other matter.  256/512, a forward with the last state and forward and backward, with the
//    scan and the streaming kernels / so: 128 heads of 2049 positions 444 / 279 and 1233 / 996, of 8192 1479 / 1047 and 4318 / 3671,
//    512 of 1024 779 / 557 and 1994 / 1797, 1024 of 512 816 / 602 and 1726 / 1678.
int columns(const ChainHvArgs& a, int BH) {
  if (a.DHQK != 64 && a.DHQK != 128 && a.DHQK != 256) return 0;
  if (((size_t)a.S + kStep) * (size_t)(a.DHHV > a.DHQK ? a.DHHV : a.DHQK) * 2 >= ((size_t)1 << 32)) return 0;  // 32-bit offsets in a head
  if (a.S <= 2 * kChunk) return 0;
  // (dV reads no V; the kept states read no Q and write no rows)
  if (((uintptr_t)a.Q | (uintptr_t)a.K | (uintptr_t)(a.dH != nullptr ? a.dH : a.V) | (uintptr_t)a.Out) % 16 != 0) return 0;
  const int cus = device_cu_count();
  if (cus <= 0) return 0;
  auto full = [&](int w, int pct) {
    const long long n = (long long)BH * (a.DHHV / w), rounds = (n + cus - 1) / cus;
    return a.DHHV % w == 0 && 100 * n >= pct * rounds * cus;
  };
  if (full(256, 85)) return 256;
  if (full(128, 95) && !(a.DHQK == 256 && a.DHHV % 512 == 0)) return 128;
  return 0;
}
}  // namespace

bool chain_hv_preferred(const ChainHvArgs& a, int BH) { return columns(a, BH) != 0; }

static const char* launch(const ChainHvArgs& a, int BH, int kind, hipStream_t stream) {
  if (a.stride < 1 || a.stride > kMaxStateStride) return "chain_hv: state stride out of range";
  switch (columns(a, BH) * 1000 + a.DHQK) {
    case 256256: return launch_w<256, 256>(a, BH, kind, stream);
    case 256128: return launch_w<128, 256>(a, BH, kind, stream);
    case 256064: return launch_w<64, 256>(a, BH, kind, stream);
    case 128256: return launch_w<256, 128>(a, BH, kind, stream);
    case 128128: return launch_w<128, 128>(a, BH, kind, stream);
    case 128064: return launch_w<64, 128>(a, BH, kind, stream);
    default: return "chain_hv: unsupported shape";
  }
}
const char* launch_chain_hv(const ChainHvArgs& a, int BH, bool is_dv, hipStream_t stream) {
  return launch(a, BH, is_dv ? kBackward : kForward, stream);
}
const char* launch_chain_states(const ChainHvArgs& a, int BH, hipStream_t stream) { return launch(a, BH, kKeptStates, stream); }

}  // namespace mlstm
