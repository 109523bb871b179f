// dQ and dK of the chunkwise backward for the default state stride of 2, organised around the window of two chunks
// that share a kept state: the same arithmetic as par_qk.hip (see there for the formulas and the state-stride
// algebra), arranged so that every operand passes through a CU as few times as the register file allows and the
// score blocks are computed once for both gradients.
//
// With c0 = 2s, c1 = 2s + 1 the two chunks of window s (256 positions, t and j counted over the window), C the state
// kept before c0 and dC the state kept after c1:
//   P[t][j]   = exp(u_t - w_j + G) / sqrt(DHQK) * rho_t * (dH_t . v_j)   for j <= t   (G = decay of c0 when t is in
//               c1 and j in c0, else 0): a lower triangle of 8 x 8 blocks of 32 x 32, 36 blocks, kept in LDS as bf16
//   dQ[t][:]  = csq_t * (C dH_t)  + sum_j P[t][j] k_j
//   dK[j][:]  = csk_j * (dC v_j)  + sum_t P[t][j] q_t
//
//   * One PERSISTENT workgroup per CU (twelve waves) walks its share of the windows.  Four PRODUCER waves move data
//     only, in slabs of 32 KB through a FIFO of two register sets into a ring of two LDS slots; eight CONSUMER waves
//     read operand fragments from LDS, multiply, gate and write the results.  One barrier per slab.
//   * Three phases per window, all with a static step structure (NV = DHHV / 32; written for head-dim tiles of 256: with
//     tiles of 128 and 64 a slab of rows holds 128 and 256 positions, two steps and one instead of four):
//       S  NV steps  [dH rows x 32 value columns | V rows x 32 value columns]      scores of all 36 blocks, then gating
//       Q  NV steps  [C fragments of 32 value columns | dH rows x 32 columns]      Out^T += C dH^T  (256 x 256 tile)
//           4 steps  [64 K rows x 256 head-dim entries]                            Out^T += K^T P^T
//           4 steps  [64 Q rows]                                                   row dots q . dQ; dQ rows leave
//       K  NV steps  [dC fragments | V rows],  4 steps [64 Q rows], 4 steps [64 K rows]   the same for dK (P read
//                                                                                  transposed)
//     A window moves 3 * DHHV + 512 KB through the CU (2048 KB at DHHV = 512) where the same arrangement for
//     single chunks and gradients took 2944 KB, and multiplies every score block once instead of twice.
//   * A consumer wave owns 64 head-dim rows x four 32-position blocks of alternating parity (128 accumulator
//     registers); the causal structure then loads both parities nearly alike.  The q (k) rows of the gate-gradient
//     row dots come through the ring like every other operand (fetched by the consumers themselves they cost a
//     memory latency per handful of positions); the rounded results pass through a private 2 KB staging tile per
//     wave into row order and are stored as full 128-byte lines.
//   * A window without a state on one side (no initial state, no gradient after the end) leaves out that phase's NV steps:
//     the state and the second reading of dH (V), a quarter of a 256/512 window.
// Supported: state stride 2, any head dimensions (multiples of 64; DHQK in tiles of 256, 128 or 64, whichever divides it).
// Measured on MI355X, us, tiled pair kernel -> this one: 128/256 with 262144 token-heads 326 -> 162, 128/128 259 -> 112,
// 64/128 244 -> 77, 64/64 with 524288 419 -> 110, 512/1024 with 32768 210 -> 180; 256/512 with 524288 1042 -> 770.
#include <type_traits>

#include "kernels.h"
#include "window.h"

namespace mlstm {
namespace {
constexpr int kWqVecOfs = kWinPOfs + kWinPBytes;  // u[256], w[256], lqr[256] (fp32)
constexpr int kWqRedOfs = kWqVecOfs + 3 * 1024;   // [4][256] row-dot partials per 64-row block of the head dimension
constexpr int kWqStgOfs = kWqRedOfs + 4 * 1024;   // [8 waves][16 rows][64 elements] staging tiles
constexpr int kWqCsOfs = kWqStgOfs + 8 * 2048;    // [256] column scale of the inter-chunk part of the running phase
constexpr int kWqSmem = kWqCsOfs + 1024;
static_assert(kWqSmem <= 160 * 1024, "LDS budget of one CU");

// The order of the windows.  Those of a head that have a phase less, because the state in front of the first or behind the last
// one is known to be zero, come last, so that the rounds of the workgroups end together.  In the round in which they begin
// neighbours lie on different XCDs: every XCD having a range of its own, as in the other rounds, they would all fall to the last
// ones.  Us, as they come / last / last and dealt: 32 heads of 16384 positions, 256/512, 791 / 774 / 777, 128 of 1024 196 / - / 190,
// 64 of 1000 95 / 102 / 94; tiles of 128 rows gain nothing (128/256, 128 of 2048, 164 / - / 166) and keep the order.
struct QkOrder {
  int G, n_items, NWIN, own, dealt;
  int lo, hi, n_full;  // windows lo .. hi - 1 of a head have everything to do; how many of all heads
  __device__ __forceinline__ QkOrder(int b, int G_, int n, int w, bool first, bool last) : G(G_), n_items(n), NWIN(w) {
    own = G % 8 == 0 ? (b % 8) * (G / 8) + b / 8 : b;  // consecutive places share an XCD (and its L2)
    dealt = b;
    lo = first ? 1 : 0;
    hi = max(last ? NWIN - 1 : NWIN, lo);
    n_full = n_items / NWIN * (hi - lo);
  }
  // the item of this workgroup in round `round`; the assignment rotates by one per round
  __device__ __forceinline__ bool item(WinItem& it, int round) const {
    const bool mixed = n_full < n_items && round == n_full / G && n_full % G != 0;
    const long long idx = (long long)round * G + (mixed ? dealt : (own + round) % G);
    if (idx >= n_items) return false;
    const int i = (int)idx, full = hi - lo;
    if (i < n_full) {
      it.win = lo + i % full;
      it.bh = i / full;
    } else {
      const int per = NWIN - full, j = (i - n_full) % per;
      it.win = j < lo ? j : hi + j - lo;
      it.bh = (i - n_full) / per;
    }
    return true;
  }
};
}  // namespace

// DT = head-dim rows of a tile: 256, 128 or 64.  MULTI: the head dimension is several tiles, walked one after the other
// with the same scores (otherwise it is a compile-time constant).
// RAGGED: S is not a multiple of 256 (at compile time: the clamps and predicated stores cost full windows 1 %).
template <int DT, bool MULTI, bool RAGGED, bool F16>
__global__ __launch_bounds__(768) void window_qk_kernel(ParQkArgs a, int n_items, int n_rounds, int n_bh) {
  constexpr int NDI = DT / 64;           // consumer waves over the head-dim rows of a tile
  constexpr int NPG = 8 / NDI;           // consumer waves over the positions: blocks NPG * nb + pg of 32 positions
  constexpr int NNB = NDI;               // position blocks per wave
  constexpr int ZROWS = 16384 / DT;      // positions per slab of K / Q rows
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* const uvec = (float*)(smem_raw + kWqVecOfs);  // [256] u_t of the window's positions
  float* const wvec = uvec + 256;                      // [256] w_j
  float* const lqr = wvec + 256;                       // [256] log2(rho_t / sqrt(DHQK))
  float* const red = (float*)(smem_raw + kWqRedOfs);
  float* const csv = (float*)(smem_raw + kWqCsOfs);

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int G = gridDim.x;
  const int NC = a.NC, S = a.S, DHHV = a.DHHV, DHQK = MULTI ? a.DHQK : DT;
  const int ND = DHQK / 16, NDG = DHQK / DT;
  const int NV = DHHV / 32;   // steps of 32 value columns (even)
  const int NWIN = (NC + 1) / 2;  // the last window may hold one chunk only: the other half of it is past the end
  const size_t Sp = (size_t)NC * kChunk;
  // no initial state, no gradient after the last chunk: the steps that would multiply them fall away
  const bool zero_c = __builtin_amdgcn_readfirstlane(*a.g.zero_c) != 0, zero_dc = a.zero_dc != 0;
  const QkOrder order(blockIdx.x, G, n_items, NWIN, DT == 256 && zero_c, DT == 256 && zero_dc);

  if (wave_all >= 8) {
    // =========================================================================================== producer waves
    // Load step L (counted over all windows of this workgroup) uses register set L & 1 and ring slot L & 1.  Handling
    // it means: pass barrier L - 3, write slab L - 2 from the register set to LDS, request slab L into the set.  The
    // destination in LDS travels with the data: 16-byte-unit offsets of the first piece of either half of the slab
    // (pieces 0..3 and 4..7, 4096 bytes apart inside a half).
    const int p = (wave_all - 8) * 64 + lane;  // 0 .. 255: every thread moves eight 16-byte pieces of every slab
    u32x4 fd0[8], fd1[8];
    uint32_t fw0 = 0, fw1 = 0;
    int L = 0, passed = 0;  // load steps; barriers passed
#define WQ_BARRIER                                                                                                   \
  if (L - 2 > passed) {                                                                                              \
    __syncthreads();                                                                                                 \
    ++passed;                                                                                                        \
  }
#define WQ_STORE(E)                                                                                                  \
  {                                                                                                                  \
    const uint32_t w_ = fw##E;                                                                                       \
    const uint32_t dA_ = (w_ & 0xFFFFu) * 16, dB_ = (w_ >> 16) * 16;                                                 \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) *(u32x4*)(smem_raw + dA_ + i_ * 4096) = fd##E[i_];              \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) *(u32x4*)(smem_raw + dB_ + i_ * 4096) = fd##E[4 + i_];          \
  }
    // one step: bA_/gA_/sA_ base, first byte offset and piece distance of pieces 0..3, bB_/gB_/sB_ of pieces 4..7;
    // nA_ pieces of the first half that carry something (small state slabs; the rest lands where nobody reads);
    // lA_, lB_ largest byte offset of a piece (rows past the end of the sequence re-read its last row: their score
    // factors are zero and their results are not stored), dAu_ / dBu_ destination units of the two halves inside the slot
#define WQ_PROC(E, bA_, gA_, sA_, lA_, nA_, bB_, gB_, sB_, lB_, dAu_, dBu_)                                                         \
  {                                                                                                                  \
    WQ_BARRIER                                                                                                       \
    /* piece by piece: the old content of a register goes to LDS, then the register is requested anew, so that the */ \
    /* LDS port and the vector-memory path of the CU work side by side instead of one after the other */             \
    const uint32_t w_ = fw##E;                                                                                       \
    const uint32_t oA_ = (w_ & 0xFFFFu) * 16, oB_ = (w_ >> 16) * 16;                                                 \
    const bool st_ = L >= 2;                                                                                         \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) {                                                               \
      if (st_) *(u32x4*)(smem_raw + oA_ + i_ * 4096) = fd##E[i_];                                                    \
      if (i_ < (nA_)) fd##E[i_] = *(const u32x4*)((bA_) + (RAGGED ? min((gA_) + i_ * (sA_), (lA_)) : (gA_) + i_ * (sA_)));                                                     \
    }                                                                                                                \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) {                                                               \
      if (st_) *(u32x4*)(smem_raw + oB_ + i_ * 4096) = fd##E[4 + i_];                                                \
      fd##E[4 + i_] = *(const u32x4*)((bB_) + (RAGGED ? min((gB_) + i_ * (sB_), (lB_)) : (gB_) + i_ * (sB_)));                                                 \
    }                                                                                                                \
    fw##E = ((dAu_) + (E) * (kWinSlot / 16)) | (((dBu_) + (E) * (kWinSlot / 16)) << 16);                               \
    ++L;                                                                                                             \
  }
    WinItem it;
    for (int rd = 0; rd < n_rounds; ++rd) {
      if (!order.item(it, rd)) continue;
      const uint32_t pl = (uint32_t)opaque(p);
      const char* const dH_b = (const char*)a.dH + (size_t)it.bh * S * DHHV * 2;
      const char* const V_b = (const char*)a.V + (size_t)it.bh * S * DHHV * 2;
      const char* const K_b = (const char*)a.K + (size_t)it.bh * S * DHQK * 2;
      const char* const Q_b = (const char*)a.Q + (size_t)it.bh * S * DHQK * 2;
      const size_t st_ofs = ((size_t)it.bh * NWIN + it.win) * (size_t)(DHHV / 32) * ND * 1024;
      const char* const C_b = (const char*)a.states + st_ofs;
      const char* const dC_b = (const char*)a.states2 + st_ofs;
      const uint32_t t0 = (uint32_t)it.win * 256;  // first position of the window
      // operand rows x 32 value columns: piece (row, unit) = (pl / 4 + 64 i, pl % 4), 64 bytes per row and slab
      const uint32_t xrow = pl >> 2, xun = pl & 3;
      const uint32_t xdu = xrow * 4 + (xun ^ (uint32_t)win_f64((int)xrow));
      const uint32_t xg = (t0 + xrow) * (uint32_t)(DHHV * 2) + xun * 16;
      const uint32_t xstep = 64 * (uint32_t)DHHV * 2;
      const uint32_t xlim = (uint32_t)(S - 1) * (uint32_t)(DHHV * 2) + xun * 16;  // this thread's unit of the last row
      // state fragments of 32 value columns: DT / 16 KB contiguous in memory; lanes 32..63 of every fragment are stored 4 slots off
      // and every second fragment 8, so that the two lane halves of two fragments that a transposing read touches together fall
      // on different LDS banks
      const uint32_t cdu = pl ^ (((pl >> 5) & 1) << 2) ^ (((pl >> 6) & 1) << 3);
      // ZROWS rows x DT head-dim entries: piece (row, unit) = (pl / UPR + 256 / UPR i, pl % UPR)
      constexpr int UPR = DT / 8;  // 16-byte units per row of a tile
      const uint32_t zpitch = (uint32_t)DHQK * 2;
      const uint32_t zrow = pl / UPR, zun = pl % UPR;
      const uint32_t zdu = zrow * UPR + (zun ^ (uint32_t)win_zsw<DT * 2>((int)zrow));
      const uint32_t zg0 = (t0 + zrow) * zpitch + zun * 16;
      const uint32_t zlim0 = (uint32_t)(S - 1) * zpitch + zun * 16;
      const uint32_t zstep = (256 / UPR) * zpitch;
      // (every loop works on its own opaque copy of the offsets: addresses shared between two loops would otherwise be
      // kept, and spilled, across everything in between)
#define WQ_ROW_SLAB(E, b_, z_)                                                                                       \
  WQ_PROC(E, b_, zz + (uint32_t)((z_) * ZROWS) * zpitch, zstep, zlim, 4, b_,                                         \
          zz + (uint32_t)((z_) * ZROWS) * zpitch + 4 * zstep, zstep, zlim, zdu, 1024 + zdu)
    // the rows of the products (first) and those of the row dots
#define WQ_ROWS(bA_, bB_)                                                                                            \
  {                                                                                                                  \
    const uint32_t zz = (uint32_t)opaque((int)zg), zlim = (uint32_t)opaque((int)zl);                                 \
    if constexpr (NDI == 1) {                                                                                        \
      WQ_ROW_SLAB(0, bA_, 0)                                                                                         \
      WQ_ROW_SLAB(1, bB_, 0)                                                                                         \
    } else {                                                                                                         \
      for (int z = 0; z < NDI; z += 2) {                                                                             \
        WQ_ROW_SLAB(0, bA_, z)                                                                                       \
        WQ_ROW_SLAB(1, bA_, z + 1)                                                                                   \
      }                                                                                                              \
      for (int z = 0; z < NDI; z += 2) {                                                                             \
        WQ_ROW_SLAB(0, bB_, z)                                                                                       \
        WQ_ROW_SLAB(1, bB_, z + 1)                                                                                   \
      }                                                                                                              \
    }                                                                                                                \
  }
      // ---- gate vectors of the window: requested in front of its first slab, in LDS two steps later, when the consumers are in the
      // last step of the window before, which reads none of them any more.  (As requests of the consumer waves each phase
      // waited for them, and with them for the stores of the phase before.  256 heads of 2048, 64/64: 123 -> 111 us; 128 heads,
      // 128/256: 164.6 -> 161.5; 32 heads of 16384, 256/512: 783 -> 774; with two windows per workgroup of 256/256 1 % more.)
      const int n_pos = RAGGED ? S - 256 * it.win : 256, c0 = 2 * it.win;
      // keys of c0 see dC through chunk c1, where there is one (the gradient kept is that after the last chunk); positions of c1 see
      // C through chunk c0
      const bool two = !RAGGED || c0 + 1 < NC;
      float pu, pw, pr, pb, pa, pg0, pg1, pm0, pm1, pm2, csq, csk;
      {
        const size_t gi = (size_t)it.bh * Sp + (size_t)c0 * kChunk + (RAGGED ? min((int)pl, n_pos - 1) : (int)pl);
        const float* const graw = a.g.graw + (size_t)it.bh * NC + c0;
        const float* const mst = a.g.mstates + (size_t)it.bh * (NC + 1) + c0;
        pg0 = graw[0];
        pg1 = graw[two ? 1 : 0];
        pm0 = mst[0];
        pm1 = mst[1];
        pm2 = mst[two ? 2 : 1];
        pu = a.g.u[gi];
        pw = a.g.w[gi];
        pr = (a.use_nrow ? a.nrow : a.g.u)[gi];
        pb = a.g.bbar[gi];
        pa = a.g.abar[gi];
      }
      // ---- phase S: dH rows | V rows
      {
        const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim);
        WQ_PROC(0, dH_b, xx, xstep, xl, 4, V_b, xx, xstep, xl, xdu, 1024 + xdu)
        WQ_PROC(1, dH_b, xx + 64, xstep, xl + 64, 4, V_b, xx + 64, xstep, xl + 64, xdu, 1024 + xdu)
      }
      WQ_BARRIER
      {
        // past the end: no key (w = infinity), no query (factor 0)
        const int t = (int)pl;
        const bool in = !RAGGED || t < n_pos;
        const float rh = a.use_nrow ? 1.f / (pr + a.eps) : 1.f;
        uvec[t] = pu;
        wvec[t] = in ? pw : __builtin_inff();
        lqr[t] = in ? __log2f(a.qk_scale * rh) : -__builtin_inff();
        csq = pb * a.qk_scale * rh * (t >= 128 ? __expf(pg0 + pm0 - pm1) : 1.f);
        csk = pa * (t < 128 && two ? __expf(pg1 + pm1 - pm2) : 1.f);
      }
      {
        const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim);
        for (int w = 2; w < NV; w += 2) {
          WQ_PROC(0, dH_b, xx + w * 64, xstep, xl + w * 64, 4, V_b, xx + w * 64, xstep, xl + w * 64, xdu, 1024 + xdu)
          WQ_PROC(1, dH_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, 4, V_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, xdu, 1024 + xdu)
        }
      }
      for (int dg = 0; dg < NDG; ++dg) {
      const uint32_t cstep = (uint32_t)ND * 1024;  // fragments of 32 value columns, all head-dim tiles
      const uint32_t zg = zg0 + dg * (DT * 2), zl = zlim0 + dg * (DT * 2);
      // ---- phase Q: C fragments | dH rows, then the K rows (products) and the Q rows (row dots)
      {
        const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim), cc = (uint32_t)opaque((int)(pl * 16 + dg * (DT / 16) * 1024));
        const int nv = zero_c && it.win == 0 ? 0 : NV;
        for (int w = 0; w < nv; w += 2) {
          WQ_PROC(0, C_b, (uint32_t)w * cstep + cc, 4096, 0xffffffffu, NDI, dH_b, xx + w * 64, xstep, xl + w * 64, cdu, 1024 + xdu)
          WQ_PROC(1, C_b, (uint32_t)(w + 1) * cstep + cc, 4096, 0xffffffffu, NDI, dH_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, cdu, 1024 + xdu)
          if (w == 0) {
            WQ_BARRIER  // the consumers are done with the factors of the phase before
            csv[pl] = csq;
          }
        }
      }
      WQ_ROWS(K_b, Q_b)
      // ---- phase K: dC fragments | V rows, then the Q rows (products) and the K rows (row dots)
      {
        const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim), cc = (uint32_t)opaque((int)(pl * 16 + dg * (DT / 16) * 1024));
        const int nv = zero_dc && it.win == NWIN - 1 ? 0 : NV;
        for (int w = 0; w < nv; w += 2) {
          WQ_PROC(0, dC_b, (uint32_t)w * cstep + cc, 4096, 0xffffffffu, NDI, V_b, xx + w * 64, xstep, xl + w * 64, cdu, 1024 + xdu)
          WQ_PROC(1, dC_b, (uint32_t)(w + 1) * cstep + cc, 4096, 0xffffffffu, NDI, V_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, cdu, 1024 + xdu)
          if (w == 0) {
            WQ_BARRIER  // the consumers are done with the factors of the phase before
            csv[pl] = csk;
          }
        }
      }
      WQ_ROWS(Q_b, K_b)
      }
#undef WQ_ROWS
#undef WQ_ROW_SLAB
    }
    // ---- drain: the last two slabs go to LDS, then the barriers of the consumers' last steps and of the final row dots
    if (L > 0) {
      WQ_BARRIER
      WQ_STORE(0)
      __syncthreads();
      WQ_STORE(1)
      __syncthreads();
      __syncthreads();
    }
#undef WQ_PROC
#undef WQ_BARRIER
#undef WQ_STORE
  } else {
    // =========================================================================================== consumer waves
    const int wave = wave_all;
    const int tid = wave * 64 + lane;
    const int di = wave % NDI, pg = wave / NDI;  // head-dim rows 64 di .. of a tile, position blocks NPG * nb + pg
    unsigned char* const stg = smem_raw + kWqStgOfs + wave * 2048;
    const WinBlocks blk = win_blocks(wave);
    f32x16 acc[2][NNB];
    WinItem it, prev;
    prev = WinItem{0, 0};
    int pending = 0;       // row dots waiting in `red`: 1 dQ of `prev`, 2 dK of `prev`
    int prev_dg = 0;       // ... of this head-dim tile
    uint32_t slot = 0;     // ring slot of the next slab
    auto next_slab = [&]() {
      const unsigned char* s = smem_raw + slot * kWinSlot;
      slot ^= 1;
      return s;
    };
    // row dots of the last finished phase: the four 64-row blocks' partials meet in LDS, 256 threads add them up
    auto finish_rowdots = [&]() {
      if (pending && tid < 256) {
        float dot = red[tid];
        if constexpr (NDI == 2) dot += red[256 + tid];
        if constexpr (NDI == 4) dot = (dot + red[256 + tid]) + (red[512 + tid] + red[768 + tid]);
        // one slot per head-dim tile: [tile][batch * head][position]
        if (!RAGGED || prev.win * 256 + tid < S)
          (pending == 2 ? a.rowdot2 : a.rowdot)[((size_t)prev_dg * n_bh + prev.bh) * Sp + (size_t)prev.win * 256 + tid] = dot;
      }
      pending = 0;
    };

    for (int rd = 0; rd < n_rounds; ++rd) {
      if (!order.item(it, rd)) continue;
      const int bh = it.bh, c0 = 2 * it.win;
      const float* graw = a.g.graw + (size_t)bh * NC;
      const float g01 = graw[c0];   // decay over chunk c0: what separates a position of c1 from the keys of c0
      const int n_pos = RAGGED ? S - 256 * it.win : 256;   // positions of the window inside the sequence (256 or more: all)

      // ================================================================================= phase S: the score blocks
      {
        f32x16 sacc[5];
#pragma unroll
        for (int e = 0; e < 5; ++e)
#pragma unroll
          for (int i = 0; i < 16; ++i) sacc[e][i] = 0.f;
        for (int w = 0; w < NV; ++w) {
          __syncthreads();
          const unsigned char* const slab = next_slab();
          if (w == 0) {
            finish_rowdots();
            prev = it;
          }
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          const int ra = 32 * blk.ta + r, rc = 32 * blk.tc + r;
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            Frag Ba, Bc;
            Ba.u = *(const uint4*)(slab + ra * 64 + (((2 * ks + h) ^ win_f64(ra)) * 16));
            Bc.u = *(const uint4*)(slab + rc * 64 + (((2 * ks + h) ^ win_f64(rc)) * 16));
#pragma unroll
            for (int e = 0; e < 5; ++e) {
              const int jrow = 32 * (e < 3 ? blk.ja + e : blk.jc + e - 3) + r;
              Frag A;
              A.u = *(const uint4*)(slab + 16384 + jrow * 64 + (((2 * ks + h) ^ win_f64(jrow)) * 16));
              mfma32<F16>(sacc[e], A, e < 3 ? Ba : Bc);   // rows: keys j, columns: positions t
            }
          }
        }
        // ---- gating: P[t][j] = scores * exp(u_t - w_j + G) / sqrt(DHQK) * rho_t, zero above the diagonal
        {
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
#pragma unroll
          for (int e = 0; e < 5; ++e) {
            if (e < 3 + blk.nc) {
              const int tb = e < 3 ? blk.ta : blk.tc, jb = e < 3 ? blk.ja + e : blk.jc + e - 3;
              const float gg = (tb >= 4 && jb < 4) ? g01 : 0.f;
              const float un = uvec[32 * tb + r] + gg;
              const float lq = lqr[32 * tb + r];
              unsigned char* const pb = smem_raw + kWinPOfs + (tb * (tb + 1) / 2 + jb) * 2048 + r * 64;
              const int fr = win_f64(r);
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                const int j0 = 8 * g4 + 4 * h;
                const float4 wj = *(const float4*)(wvec + 32 * jb + j0);
                const float wv[4] = {wj.x, wj.y, wj.z, wj.w};
                float pv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const float e2 = __builtin_amdgcn_exp2f(__builtin_fmaf(un - wv[q], kWinLog2e, lq));
                  const bool keep = tb != jb || j0 + q <= r;
                  pv[q] = keep ? sacc[e][4 * g4 + q] * e2 : 0.f;
                }
                *(uint2*)(pb + ((g4 ^ fr) * 16) + 8 * h) = make_uint2(pack2<F16>(pv[0], pv[1]), pack2<F16>(pv[2], pv[3]));
              }
            }
          }
        }
      }

      // ============================================================================ phases Q (dQ) and K (dK)
      auto run_phase = [&](auto DKT, int dg) {
        constexpr bool dk = decltype(DKT)::value;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int nb = 0; nb < NNB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.f;

        const bool no_state = dk ? zero_dc && it.win == NWIN - 1 : zero_c && it.win == 0;
        // ---- Out^T += State Xn^T over the value columns, 32 at a time.  The stored fragments (made for a contraction
        // over the head dimension) are read with the transposing LDS read: lane i16 of a 16-lane block addresses
        // value column k0 + i16 / 4 and the 4 consecutive head-dim rows n0 + 4 (i16 % 4) .. + 3
        const int nv = no_state ? 0 : NV;
        for (int w = 0; w < nv; ++w) {
          __syncthreads();
          const unsigned char* const Cf = next_slab();
          if (w == 0) finish_rowdots();
          const unsigned char* const Xn = Cf + 16384;
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          const int q16 = (le >> 4) & 1, i16 = le & 15;
          const int d_grp = i16 & 3;
          const int h_src = d_grp & 1, a_src = d_grp >> 1;
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            Frag A[2], B[NNB];
#pragma unroll
            for (int nb = 0; nb < NNB; ++nb) {
              const int row = 32 * (NPG * nb + pg) + r;
              B[nb].u = *(const uint4*)(Xn + row * 64 + (((2 * ks + h) ^ win_f64(row)) * 16));
            }
            const int wrow = 16 * ks + 8 * h + (i16 >> 2);  // value column inside the 32-column slab (first read)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
              const int ds_l = (64 * di + 32 * mb + 16 * q16) / 16;
#pragma unroll
              for (int half = 0; half < 2; ++half) {
                const int wr = wrow + 4 * half;
                const int slot_l = (32 * h_src + wr) ^ (h_src << 2) ^ (q16 << 3);
                A[mb].d[half] = lds_read_tr16(Cf + ((size_t)ds_l * 64 + slot_l) * 16 + 8 * a_src);
              }
            }
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int nb = 0; nb < NNB; ++nb) mfma32<F16>(acc[mb][nb], A[mb], B[nb]);
          }
        }
        // column scale of the inter-chunk part (kept apart from the matrix instructions around it)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < NNB; ++nb) {
          // (without a state nothing was written there, and the accumulators are zero)
          const float cs = no_state ? 0.f : csv[32 * (NPG * nb + pg) + (opaque(lane) & 31)];
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) acc[mb][nb] *= cs;
        }
        __builtin_amdgcn_sched_barrier(0);

        // ---- Out^T += Z^T P'^T over the 256 positions of the window, ZROWS rows of Z per slab (Z = K for dQ with
        // P' = P: contraction over the keys j; Z = Q for dK with P' = P^T: contraction over the positions t)
#pragma unroll
        for (int z = 0; z < NDI; ++z) {
          __syncthreads();
          const unsigned char* const Zs = next_slab();
          if (z == 0 && no_state) finish_rowdots();
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          const int q16 = (le >> 4) & 1, i16 = le & 15;
          const int krow = 8 * h + (i16 >> 2);
          const int zun = 2 * q16 + ((i16 & 3) >> 1), zin = 8 * (i16 & 1);   // 16-byte unit and byte inside it
#pragma unroll
          for (int zh = 0; zh < ZROWS / 32; ++zh) {
            const int ob = z * (ZROWS / 32) + zh;  // 32-position block of the contraction index
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
              Frag A[2];
#pragma unroll
              for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                  const int row = 32 * zh + 16 * kk + krow + 4 * half;
                  const int un = 8 * di + 4 * mb + zun;
                  A[mb].d[half] = lds_read_tr16(Zs + row * (DT * 2) + ((un ^ win_zsw<DT * 2>(row)) * 16) + zin);
                }
#pragma unroll
              for (int nb = 0; nb < NNB; ++nb) {
                const WinSide side = win_side(dk, ob, nb, NPG);
                if (side == kWinOff) continue;
                const int nbk = NPG * nb + pg;   // the wave's position block (dQ: t, dK: j)
                const bool live = side == kWinOn || (dk ? ob >= nbk : ob <= nbk);
                // (the matrix instructions stay unconditional: accumulators that pass through a branch get copied)
                Frag Ax[2], B;
                B.u = Ax[0].u = Ax[1].u = make_uint4(0u, 0u, 0u, 0u);
                if (live) {
                  Ax[0] = A[0];
                  Ax[1] = A[1];
                  if (dk) {
                    // P^T: rows t of block (ob, nbk) are the contraction index -> transposing read
                    const unsigned char* const pb = smem_raw + kWinPOfs + (ob * (ob + 1) / 2 + nbk) * 2048;
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                      const int row = 16 * kk + krow + 4 * half;
                      B.d[half] = lds_read_tr16(pb + row * 64 + ((zun ^ win_f64(row)) * 16) + zin);
                    }
                  } else {
                    const unsigned char* const pb = smem_raw + kWinPOfs + (nbk * (nbk + 1) / 2 + ob) * 2048;
                    B.u = *(const uint4*)(pb + r * 64 + (((2 * kk + h) ^ win_f64(r)) * 16));
                  }
                }
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) mfma32<F16>(acc[mb][nb], Ax[mb], B);
              }
            }
          }
        }

        // ---- results, ZROWS positions per step: the x rows (q for dQ, k for dK) of those positions arrive as one more
        // slab; every wave owns one 32-position block of them.  Row dots sum_d x Out from the fp32 accumulators (they
        // feed a suffix sum over the whole sequence, where the rounding noise of 16-bit outputs would add up); then
        // the rounded values pass, 16 positions at a time, through the wave's private staging tile into row order and
        // leave as full 128-byte lines.
        char* const Ob = (char*)(dk ? a.Out2 : a.Out) + ((size_t)bh * S + (size_t)c0 * kChunk) * (DHQK * 2) + dg * (DT * 2);
#pragma unroll
        for (int z = 0; z < NDI; ++z) {
          __syncthreads();
          const unsigned char* const Xs = next_slab();
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          {
            const int row = 32 * pg + r;
            const unsigned char* const xrow = Xs + row * (DT * 2) + 8 * h;
            const int sw = win_zsw<DT * 2>(row);
            float part = 0.f;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                const uint2 xv = *(const uint2*)(xrow + (((8 * di + 4 * mb + g4) ^ sw) * 16));
                part += acc[mb][z][4 * g4 + 0] * lo2<F16>(xv.x);
                part += acc[mb][z][4 * g4 + 1] * hi2<F16>(xv.x);
                part += acc[mb][z][4 * g4 + 2] * lo2<F16>(xv.y);
                part += acc[mb][z][4 * g4 + 3] * hi2<F16>(xv.y);
              }
            part += __shfl_xor(part, 32);
            if (h == 0) red[di * 256 + ZROWS * z + row] = part;
          }
          const uint32_t lofs = (uint32_t)(le >> 3) * (uint32_t)(DHQK * 2) + (uint32_t)(128 * di + 16 * (le & 7));
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            if ((r >> 4) == q) {
              const int row = r & 15;
#pragma unroll
              for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4)
                  *(uint2*)(stg + row * 128 + (((4 * mb + g4) ^ (row & 7)) * 16) + 8 * h) =
                      make_uint2(pack2<F16>(acc[mb][z][4 * g4 + 0], acc[mb][z][4 * g4 + 1]),
                                 pack2<F16>(acc[mb][z][4 * g4 + 2], acc[mb][z][4 * g4 + 3]));
            }
            __builtin_amdgcn_wave_barrier();
            const int row8 = le >> 3, un = le & 7;
            const u32x4 o0 = *(const u32x4*)(stg + row8 * 128 + ((un ^ row8) * 16));
            const u32x4 o1 = *(const u32x4*)(stg + (row8 + 8) * 128 + ((un ^ row8) * 16));
            __builtin_amdgcn_wave_barrier();
            const uint32_t n0 = (uint32_t)(ZROWS * z + 32 * pg + 16 * q);
            if (!RAGGED || (int)n0 + row8 < n_pos) __builtin_nontemporal_store(o0, (u32x4*)(Ob + (lofs + n0 * (uint32_t)(DHQK * 2))));
            if (!RAGGED || (int)n0 + 8 + row8 < n_pos) __builtin_nontemporal_store(o1, (u32x4*)(Ob + (lofs + (n0 + 8) * (uint32_t)(DHQK * 2))));
          }
        }
        pending = dk ? 2 : 1;
        prev_dg = dg;
      };
      for (int dg = 0; dg < NDG; ++dg) {
        run_phase(std::false_type{}, dg);
        run_phase(std::true_type{}, dg);
      }
    }
    if (pending) {   // (a workgroup without a window passes no barrier at all, like its producers)
      __syncthreads();
      finish_rowdots();
    }
  }
}

bool window_qk_supported(const ParQkArgs& a) {
  return a.stride == 2 && a.DHQK % 64 == 0 && a.DHHV % 64 == 0;
}

namespace {
template <int DT, bool MULTI, bool RAGGED, bool F16>
const char* launch_window_qk_t(const ParQkArgs& a, int BH, hipStream_t stream) {
  const long long n_items = (long long)BH * ((a.NC + 1) / 2);
  if (n_items >= (1ll << 31)) return "window_qk: too many work items";
  if ((size_t)a.S * (size_t)(a.DHHV > a.DHQK ? a.DHHV : a.DHQK) * 2 >= ((size_t)1 << 32))
    return "window_qk: one (batch, head) slab of an input exceeds 4 GiB";
  const int cus = device_cu_count();
  if (cus <= 0) return "window_qk: cannot read the number of compute units";
  int G = (int)(n_items < cus ? n_items : cus);
  if (n_items > G && G >= 8) G -= G % 8;  // (fewer items than CUs: one each, two rounds otherwise)
  const int n_rounds = (int)((n_items + G - 1) / G);
  static LdsLimit lds;
  if (!lds.allow((const void*)window_qk_kernel<DT, MULTI, RAGGED, F16>, kWqSmem))
    return "window_qk: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((window_qk_kernel<DT, MULTI, RAGGED, F16>), dim3(G), dim3(768), kWqSmem, stream, a, (int)n_items, n_rounds, BH);
  return nullptr;
}
template <int DT, bool MULTI>
const char* launch_window_qk_d(const ParQkArgs& a, int BH, hipStream_t stream) {
  if (a.S % (2 * kChunk) != 0)
    return a.f16 ? launch_window_qk_t<DT, MULTI, true, true>(a, BH, stream) : launch_window_qk_t<DT, MULTI, true, false>(a, BH, stream);
  return a.f16 ? launch_window_qk_t<DT, MULTI, false, true>(a, BH, stream) : launch_window_qk_t<DT, MULTI, false, false>(a, BH, stream);
}
}  // namespace

// Where the window kernel is the faster one: a window is one workgroup's 26 to 64 steps, so with few windows the tiled
// kernel's eight or more workgroups per window finish first.  They meet at half a window per CU with tiles of 256 rows
// (256/512, us, window / tiled: 63 / 39 at 64 windows, 65 / 73 at 128, 109 / 135 at 256), at three eighths with 128
// (128/256: 34 / 29 at 64, 33 / 50 at 128), and with 64 the window kernel wins from one window on (17 / 25).
bool window_qk_preferred(const ParQkArgs& a, int BH) {
  if (!window_qk_supported(a)) return false;
  const long long windows = (long long)BH * ((a.NC + 1) / 2), cus = device_cu_count();
  const int DT = par_qk_head_tile(a.DHQK);
  return DT == 64 || (DT == 128 ? 8 * windows >= 3 * cus : 2 * windows >= cus);
}

const char* launch_window_qk(const ParQkArgs& a, int BH, hipStream_t stream) {
  if (!window_qk_supported(a)) return "window_qk: unsupported shape (needs state stride 2, head dimensions that are multiples of 64)";
  if (a.states2 == nullptr || a.Out2 == nullptr || a.rowdot2 == nullptr) return "window_qk: the dK operands are missing";
  // (the tile decides the layout of the row-dot slots, as for the tiled kernel)
  const int DT = par_qk_head_tile(a.DHQK);
  const bool multi = a.DHQK > DT;
  if (DT == 256) return multi ? launch_window_qk_d<256, true>(a, BH, stream) : launch_window_qk_d<256, false>(a, BH, stream);
  if (DT == 128) return multi ? launch_window_qk_d<128, true>(a, BH, stream) : launch_window_qk_d<128, false>(a, BH, stream);
  return multi ? launch_window_qk_d<64, true>(a, BH, stream) : launch_window_qk_d<64, false>(a, BH, stream);
}

}  // namespace mlstm
