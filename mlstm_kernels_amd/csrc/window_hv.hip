// H and dV for windows of two chunks (state stride 2), any head dimensions: the same arithmetic as par_hv.hip (see there
// for the formulas and the state-stride algebra), in the arrangement of window_qk.hip.
//
// With t and j counted over the 256 positions of a window, C the state kept before it and dC the one kept after it:
//   P[t][j] = exp(u_t - w_j + G) / sqrt(DHQK) * (q_t . k_j)  for j <= t,  times rho_t for dV   (36 blocks of 32 x 32, in LDS)
//   H[t][:]  = ( cs_t * (C^T q_t)  + sum_j P[t][j] v_j ) / (normaliser_t + eps)
//   dV[j][:] =   cs_j * (dC^T k_j) + sum_t P[t][j] dH_t
//
//   * One PERSISTENT workgroup per CU (twelve waves) walks its share of the windows: four PRODUCER waves move slabs of up
//     to 32 KB through a FIFO of two register sets into a ring of two LDS slots, eight CONSUMER waves multiply.  One
//     barrier per slab.
//   * Steps of a window (NS = DHQK / 32, even; the value columns are walked in groups of CW):
//       S        NS steps [Q rows x 32 head-dim entries | K rows x 32]      scores of all blocks, then gating
//       per group of CW value columns:
//       O        NS steps [state fragments of 32 entries x CW | Q (K for dV) rows x 32]    Out^T  = State^T Xn^T
//       V  max(2, CW / 64) steps [V (dH) rows x CW]                                        Out^T += Xw^T P
//     A finished tile leaves during the first step of the next window's S (of several groups: each at its end).
//   * A window whose state is known to be zero has no phase O (128 heads of 2048, 128/256: the call, forward and backward,
//     487 -> 479 us with the same in window_qk.hip, before the gate vectors went to the producers).
//   * What bounds it: HBM.  Everything a window needs passes through the CU once, only the rows of O a second time: at
//     128/256 384 KB in and 128 KB out per window where the tiled kernel moved 285 KB per 64 positions; a score block is
//     computed once for all value columns of its group's window.
// Measured on MI355X, H / dV in us, tiled kernel -> this one: 128/256 with 262144 token-heads 170 / 165 -> 99 / 94
// (4.7 / 4.9 TB/s on operands and results counted once), 128/128 180 / 163 -> 72 / 67, 64/128 113 / 102 -> 56 / 51, 64/64
// with 524288 404 / 367 -> 84 / 74, 256/256 with 131072 119 / 108 -> 78 / 73, 512/1024 with 32768 142 / 141 -> 105 / 101.
// At 256/512 the streaming kernel (stream_hv.hip, Q resident: no second reading) is as fast: 137 / 128 against 147 / 131.
#include "kernels.h"
#include "window.h"

namespace mlstm {
namespace {
constexpr int kHvVecOfs = kWinPOfs + kWinPBytes;  // u[256], w[256], lqr[256] (fp32)
constexpr int kHvCsOfs = kHvVecOfs + 3 * 1024;    // cs[256] column scale of O, cs0[256] weight of q.n, inv[256], mc[256]
constexpr int kHvRowOfs = kHvCsOfs + 4 * 1024;    // [4][256] row sums of P by key block of the own chunk
constexpr int kHvMaxDhqk = 512;
constexpr int kHvNOfs = kHvRowOfs + 4 * 1024;     // forward: n before either chunk [2][DHQK]
constexpr int kHvXOfs = kHvNOfs + 2 * kHvMaxDhqk * 4;  // NORM: sums [4][2][256]; several groups: staging tiles [8][8][128 bytes]
constexpr int kHvSmem = kHvXOfs + 8 * 1024;
static_assert(kHvSmem <= 160 * 1024, "LDS budget of one CU");
}  // namespace

// MULTI: DHHV is several groups of CW columns (P then has to outlive the epilogue of a group, which otherwise stages its
// rows in it).  NORM (forward, one group): the multi-head layer / rms norm is applied to the rows as they are rounded.
// RAGGED: S is not a multiple of 256.
template <int CW, bool MULTI, bool IS_DV, bool NORM, bool RAGGED, bool F16>
__global__ __launch_bounds__(768) void window_hv_kernel(ParHvArgs a, int n_items, int n_rounds) {
  static_assert(!(IS_DV && NORM) && !(MULTI && NORM), "the head norm belongs to the forward and needs complete rows");
  constexpr int NCI = CW / 64;                     // 64-column groups = consumer waves side by side over the columns
  constexpr int NPG = 8 / NCI;                     // consumer waves over the positions
  constexpr int NNB = 8 / NPG;                     // 32-position blocks per wave: NPG * nb + pg
  constexpr int NVS = CW / 64 < 2 ? 2 : CW / 64;   // steps of V (even)
  constexpr int VROWS = 256 / NVS;                 // positions per step of V
  constexpr int UPR = CW / 8;                      // 16-byte units per row of a V slab
  constexpr int VP = VROWS * UPR / 256;            // pieces per producer thread of a V slab (8 or 4)
  constexpr int SP = CW / 64;                      // pieces per producer thread of a step's state fragments
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* const uvec = (float*)(smem_raw + kHvVecOfs);
  float* const wvec = uvec + 256;
  float* const lqr = wvec + 256;
  float* const csv = (float*)(smem_raw + kHvCsOfs);
  float* const cs0v = csv + 256;
  float* const inv = cs0v + 256;
  float* const mcv = inv + 256;
  float* const rows = (float*)(smem_raw + kHvRowOfs);
  float* const nvec = (float*)(smem_raw + kHvNOfs);
  float* const nst = (float*)(smem_raw + kHvXOfs);

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int G = gridDim.x;
  int vid = blockIdx.x;
  if (G % 8 == 0) vid = (vid % 8) * (G / 8) + vid / 8;  // consecutive ids share an XCD (and its L2)
  const int NC = a.NC, S = a.S, DHHV = a.DHHV, DHQK = a.DHQK;
  const int NS = DHQK / 32, ND = DHQK / 16, NG = MULTI ? DHHV / CW : 1;
  const int NWIN = (NC + 1) / 2;  // the last window may hold one chunk only
  const size_t Sp = (size_t)NC * kChunk;
  // without a state in front of the first window (behind the last one) phase O has nothing to add there and falls away; its
  // q . n moves to the rows of phase S.  (Such windows are not dealt out last: 128 heads of 2048, 128/256, H 116 -> 119 us, dV
  // 92 -> 99.)
  const int zero_win = a.zero_state ? (IS_DV ? NWIN - 1 : 0) : -1;

  if (wave_all >= 8) {
    // =========================================================================================== producer waves
    // Load step L uses register set and ring slot L & 1: pass barrier L - 3, write slab L - 2 from the set to LDS, request
    // slab L into it.  The destination travels with the data: byte offset of the first piece of either half of the slab,
    // further pieces 4096 bytes apart; bit 0 of the second: store in fragment order (two halves of 8 bytes, the second
    // one unit further: inside 16 head-dim entries, entry 8a + 4h + c goes to 8h + 4a + c, the order the state fragments
    // have them in).
    const int p = (wave_all - 8) * 64 + lane;
    u32x4 fd0[8], fd1[8];
    uint32_t fa0 = 0, fb0 = 0, fa1 = 0, fb1 = 0;
    int L = 0, passed = 0;  // load steps; barriers passed
#define WH_BARRIER                                                                                                   \
  if (L - 2 > passed) {                                                                                              \
    __syncthreads();                                                                                                 \
    ++passed;                                                                                                        \
  }
#define WH_PUT_B(E, i_, perm_)                                                                                       \
  {                                                                                                                  \
    if (perm_) {                                                                                                     \
      *(uint2*)(smem_raw + (oB_ + (i_) * 4096)) = make_uint2(fd##E[4 + (i_)][0], fd##E[4 + (i_)][1]);                \
      *(uint2*)(smem_raw + ((oB_ ^ 16u) + (i_) * 4096)) = make_uint2(fd##E[4 + (i_)][2], fd##E[4 + (i_)][3]);        \
    } else {                                                                                                         \
      *(u32x4*)(smem_raw + (oB_ + (i_) * 4096)) = fd##E[4 + (i_)];                                                   \
    }                                                                                                                \
  }
#define WH_STORE(E)                                                                                                  \
  {                                                                                                                  \
    const bool perm_ = __builtin_amdgcn_readfirstlane((int)(fb##E & 1)) != 0;                                        \
    const uint32_t oA_ = fa##E, oB_ = fb##E & ~1u;                                                                   \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) *(u32x4*)(smem_raw + oA_ + i_ * 4096) = fd##E[i_];              \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) WH_PUT_B(E, i_, perm_)                                          \
  }
    // nA_ / nB_ pieces of either half that carry something (the others re-request the last one of them, a cache hit that
    // lands where nobody reads); lA_, lB_: largest byte offset (rows past the end re-read the last row)
#define WH_PROC(E, bA_, gA_, sA_, lA_, nA_, bB_, gB_, sB_, lB_, nB_, dA_, dB_)                                       \
  {                                                                                                                  \
    WH_BARRIER                                                                                                       \
    /* piece by piece: the old content of a register goes to LDS, then the register is requested anew */             \
    const bool perm_ = __builtin_amdgcn_readfirstlane((int)(fb##E & 1)) != 0;                                        \
    const uint32_t oA_ = fa##E, oB_ = fb##E & ~1u;                                                                   \
    const bool st_ = L >= 2;                                                                                         \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) {                                                               \
      if (st_) *(u32x4*)(smem_raw + oA_ + i_ * 4096) = fd##E[i_];                                                    \
      if (i_ < (nA_)) fd##E[i_] = *(const u32x4*)((bA_) + (RAGGED ? min((gA_) + i_ * (sA_), (lA_)) : (gA_) + i_ * (sA_)));                           \
    }                                                                                                                \
    _Pragma("unroll") for (int i_ = 0; i_ < 4; ++i_) {                                                               \
      if (st_) WH_PUT_B(E, i_, perm_)                                                                                \
      if (i_ < (nB_)) fd##E[4 + i_] = *(const u32x4*)((bB_) + (RAGGED ? min((gB_) + i_ * (sB_), (lB_)) : (gB_) + i_ * (sB_)));                       \
    }                                                                                                                \
    fa##E = (dA_) + (E) * kWinSlot;                                                                                  \
    fb##E = (dB_) + (E) * kWinSlot;                                                                                  \
    ++L;                                                                                                             \
  }
    WinItem it;
    for (int rd = 0; rd < n_rounds; ++rd) {
      if (!win_decode(it, rd, vid, G, n_items, NWIN)) continue;
      const uint32_t pl = (uint32_t)opaque(p);
      const char* const Q_b = (const char*)a.Q + (size_t)it.bh * S * DHQK * 2;
      const char* const K_b = (const char*)a.K + (size_t)it.bh * S * DHQK * 2;
      const char* const Xn_b = IS_DV ? K_b : Q_b;
      const char* const Xw_b = (const char*)(IS_DV ? a.dH : a.V) + (size_t)it.bh * S * DHHV * 2;
      const char* const St_b = (const char*)a.states + ((size_t)it.bh * NWIN + it.win) * (size_t)(DHHV / 32) * ND * 1024;
      const uint32_t t0 = (uint32_t)it.win * 256;
      // rows x 32 head-dim entries: piece (row, unit) = (pl / 4 + 64 i, pl % 4), 64 bytes per row and slab
      const uint32_t xrow = pl >> 2, xun = pl & 3;
      const uint32_t pitch = (uint32_t)DHQK * 2;
      const uint32_t xg = (t0 + xrow) * pitch + xun * 16, xstep = 64 * pitch, xlim = (uint32_t)(S - 1) * pitch + xun * 16;
      const uint32_t xd = (xrow * 4 + (xun ^ (uint32_t)win_f64((int)xrow))) * 16;
      const uint32_t xdp = ((xrow * 4 + ((xun & 2) ^ (uint32_t)win_f64((int)xrow))) * 16 + 8 * (xun & 1)) | 1u;
      // ---- gate vectors and normaliser state of the window: requested in front of its first slab, in LDS two steps later, when
      // the consumers are in the last step of the window before, which reads none of them any more.  These waves have the
      // registers for it.  Held by the consumers until the window began they were spilled, and reading them back waited for
      // the stores of the tile that leaves there (128 heads of 2048, 128/256: H 120 -> 99 us, dV 106 -> 94; 256 heads of 2048,
      // 64/64: 92 -> 84, 81 -> 74; 64 heads of 2048, 256/256: 87 -> 78, 81 -> 74).
      const int n_pos = RAGGED ? S - 256 * it.win : 256, c0 = 2 * it.win;
      float pu, pw, pr, pc, pm = 0.f, pg, m0, m1, np[4][3];
      {
        const size_t gi = (size_t)it.bh * Sp + (size_t)c0 * kChunk + (RAGGED ? min((int)pl, n_pos - 1) : (int)pl);
        // dV: keys of the first chunk see dC through the second, where there is one; H: positions of the second see C through the
        // first
        const int cx = IS_DV && (!RAGGED || c0 + 1 < NC) ? c0 + 1 : c0;
        pg = a.g.graw[(size_t)it.bh * NC + cx];
        m0 = a.g.mstates[(size_t)it.bh * (NC + 1) + cx];
        m1 = a.g.mstates[(size_t)it.bh * (NC + 1) + cx + 1];
        pu = a.g.u[gi];
        pw = a.g.w[gi];
        if (IS_DV) {
          pr = (a.use_nrow ? a.nrow : a.g.u)[gi];
          pc = a.g.abar[gi];
        } else {
          pc = a.g.bbar[gi];
          pm = a.g.mcomb[gi];
          // n before either chunk as three partial vectors (their sum carries the full fp32 precision); entries past the end repeat
          // the last one, without a normaliser any readable word does
          const float* const n_b = a.use_nrow ? a.nstates + ((size_t)it.bh * NC + c0) * 3 * DHQK : a.g.graw;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int e = min((int)pl + 256 * i, 2 * DHQK - 1), ch = e >= DHQK ? 1 : 0;
            const int o = a.use_nrow ? (c0 + ch < NC ? ch * 3 * DHQK : 0) + e - ch * DHQK : 0, st = a.use_nrow ? DHQK : 0;
#pragma unroll
            for (int x = 0; x < 3; ++x) np[i][x] = n_b[o + x * st];
          }
        }
      }
      const uint32_t xx0 = (uint32_t)opaque((int)xg), xl0 = (uint32_t)opaque((int)xlim);
      WH_PROC(0, Q_b, xx0, xstep, xl0, 4, K_b, xx0, xstep, xl0, 4, xd, 16384 + xd)
      WH_PROC(1, Q_b, xx0 + 64, xstep, xl0 + 64, 4, K_b, xx0 + 64, xstep, xl0 + 64, 4, xd, 16384 + xd)
      WH_BARRIER
      {
        // past the end: no key (w = infinity), no query (factor 0)
        const int t = (int)pl;
        const bool in = !RAGGED || t < n_pos;
        const float f = IS_DV && a.use_nrow ? 1.f / (pr + a.eps) : 1.f, xs = __expf(pg + m0 - m1);
        uvec[t] = pu;
        wvec[t] = in ? pw : __builtin_inff();
        lqr[t] = in ? __log2f(a.qk_scale * f) : -__builtin_inff();
        if (IS_DV) {
          csv[t] = pc * (t < 128 && (!RAGGED || c0 + 1 < NC) ? xs : 1.f);
        } else {
          const float pb = pc * a.qk_scale;
          csv[t] = pb * (t >= 128 ? xs : 1.f);
          cs0v[t] = pb;
          mcv[t] = pm;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (t + 256 * i < 2 * DHQK) nvec[t + 256 * i] = (np[i][0] + np[i][1]) + np[i][2];
        }
      }
      {
        const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim);
        for (int w = 2; w < NS; w += 2) {
          WH_PROC(0, Q_b, xx + w * 64, xstep, xl + w * 64, 4, K_b, xx + w * 64, xstep, xl + w * 64, 4, xd, 16384 + xd)
          WH_PROC(1, Q_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, 4, K_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, 4,
                  xd, 16384 + xd)
        }
      }
      for (int cg = 0; cg < NG; ++cg) {
        {
          // state fragments: piece i of the thread is fragment (pl / 64 + 4 i) of the slab: column block / 2, contraction step % 2
          const uint32_t xx = (uint32_t)opaque((int)xg), xl = (uint32_t)opaque((int)xlim);
          const uint32_t f0 = pl >> 6;
          const uint32_t sg = (((uint32_t)cg * (CW / 32) + (f0 >> 1)) * ND + (f0 & 1)) * 1024 + (pl & 63) * 16;
          const uint32_t ss = 2 * (uint32_t)ND * 1024;
          const int ns = it.win == zero_win ? 0 : NS;
          for (int w = 0; w < ns; w += 2) {
            WH_PROC(0, St_b, sg + w * 2048, ss, 0xffffffffu, SP, Xn_b, xx + w * 64, xstep, xl + w * 64, 4, pl * 16, 16384 + xdp)
            WH_PROC(1, St_b, sg + (w + 1) * 2048, ss, 0xffffffffu, SP, Xn_b, xx + (w + 1) * 64, xstep, xl + (w + 1) * 64, 4,
                    pl * 16, 16384 + xdp)
          }
        }
        {
          // V rows: piece (row, unit) = (pl / UPR + 256 / UPR i, pl % UPR); the pieces of both halves are 4096 bytes apart
          const uint32_t vrow = pl / UPR, vun = pl % UPR;
          const uint32_t vp = (uint32_t)DHHV * 2, vcol = (uint32_t)cg * (CW * 2) + vun * 16;
          const uint32_t vlim = (uint32_t)(S - 1) * vp + vcol, vstep = (256 / UPR) * vp;
          const uint32_t vd = (vrow * UPR + (vun ^ (uint32_t)win_zsw<CW * 2>((int)vrow))) * 16;
          const uint32_t vg = (t0 + vrow) * vp + vcol;
          for (int z = 0; z < NVS; z += 2) {
            const uint32_t g0 = vg + (uint32_t)(z * VROWS) * vp, g1 = vg + (uint32_t)((z + 1) * VROWS) * vp;
            WH_PROC(0, Xw_b, g0, vstep, vlim, 4, Xw_b, g0 + 4 * vstep, vstep, vlim, VP - 4, vd, 16384 + vd)
            WH_PROC(1, Xw_b, g1, vstep, vlim, 4, Xw_b, g1 + 4 * vstep, vstep, vlim, VP - 4, vd, 16384 + vd)
          }
        }
      }
    }
    // ---- drain: the last two slabs go to LDS, then the barriers of the consumers' last steps and of the last epilogue
    if (L > 0) {
      WH_BARRIER
      WH_STORE(0)
      __syncthreads();
      WH_STORE(1)
      __syncthreads();
      __syncthreads();
    }
#undef WH_PROC
#undef WH_BARRIER
#undef WH_STORE
#undef WH_PUT_B
  } else {
    // =========================================================================================== consumer waves
    const int wave = wave_all;
    const int tid = wave * 64 + lane;
    const int ci = wave % NCI, pg = wave / NCI;
    constexpr int SROWS = MULTI ? 8 : 32;  // positions staged at a time (P is free between the V and the S phase)
    unsigned char* const stg = smem_raw + (MULTI ? kHvXOfs : kWinPOfs) + wave * (SROWS * 128);
    const WinBlocks blk = win_blocks(wave);
    f32x16 acc[2][NNB];
    WinItem it, prev;
    prev = WinItem{0, 0};
    bool pending = false;  // `acc` holds a finished tile of window `prev`, column group `prev_cg`
    int prev_cg = 0;
    uint32_t slot = 0;
    auto next_slab = [&]() {
      const unsigned char* s = smem_raw + slot * kWinSlot;
      slot ^= 1;
      return s;
    };
    // (normalise,) round and store the tile: 32 positions x 64 columns at a time through the wave's private staging tile
    // into row order, full 128-byte lines.  A macro: the accumulator indices stay literal.
#define WH_EPILOGUE                                                                                                  \
  {                                                                                                                  \
    const int le = opaque(lane);                                                                                     \
    const int r = le & 31, h = le >> 5;                                                                              \
    const int n_pos_ = RAGGED ? S - 256 * prev.win : 256;                                                                           \
    char* const Ob_ = (char*)a.Out + ((size_t)prev.bh * S + (size_t)prev.win * 256) * (DHHV * 2);                    \
    const uint32_t lofs_ = (uint32_t)(le >> 3) * (uint32_t)(DHHV * 2) + (uint32_t)(prev_cg * CW * 2 + 128 * ci + 16 * (le & 7)); \
    _Pragma("unroll") for (int nb = 0; nb < NNB; ++nb) {                                                             \
      const int t_ = 32 * (NPG * nb + pg) + r;                                                                       \
      float iv_ = IS_DV ? 1.f : inv[t_], sh_ = 0.f;                                                                  \
      if constexpr (NORM) {                                                                                          \
        float t1_ = 0.f, t2_ = 0.f;                                                                                  \
        _Pragma("unroll") for (int c_ = 0; c_ < NCI; ++c_) {                                                         \
          t1_ += nst[c_ * 512 + t_];                                                                                 \
          t2_ += nst[c_ * 512 + 256 + t_];                                                                           \
        }                                                                                                            \
        const float ex_ = t1_ * iv_ * (1.f / CW), ex2_ = t2_ * iv_ * iv_ * (1.f / CW);                               \
        const float mean_ = a.head_norm == 1 ? ex_ : 0.f;                                                            \
        const float rstd_ = rsqrtf(fmaxf(ex2_ - mean_ * mean_, 0.f) + a.norm_eps);                                   \
        if (ci == 0 && h == 0 && t_ < n_pos_) {                                                                      \
          const size_t tg_ = (size_t)prev.bh * S + (size_t)prev.win * 256 + t_;                                      \
          a.norm_mean[tg_] = mean_;                                                                                  \
          a.norm_rstd[tg_] = rstd_;                                                                                  \
        }                                                                                                            \
        iv_ *= rstd_;                                                                                                \
        sh_ = -mean_ * rstd_;                                                                                        \
      }                                                                                                              \
      _Pragma("unroll") for (int sr = 0; sr < 32; sr += SROWS) {                                                     \
        if (SROWS == 32 || (r & ~(SROWS - 1)) == sr) {                                                               \
          unsigned char* const srow_ = stg + (r & (SROWS - 1)) * 128 + 8 * h;                                        \
          _Pragma("unroll") for (int mb = 0; mb < 2; ++mb) _Pragma("unroll") for (int g4 = 0; g4 < 4; ++g4)          \
            *(uint2*)(srow_ + (((4 * mb + g4) ^ (r & 7)) * 16)) =                                                    \
                make_uint2(pack2<F16>(__builtin_fmaf(acc[mb][nb][4 * g4 + 0], iv_, sh_),                             \
                                      __builtin_fmaf(acc[mb][nb][4 * g4 + 1], iv_, sh_)),                            \
                           pack2<F16>(__builtin_fmaf(acc[mb][nb][4 * g4 + 2], iv_, sh_),                             \
                                      __builtin_fmaf(acc[mb][nb][4 * g4 + 3], iv_, sh_)));                           \
        }                                                                                                            \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                       \
        __builtin_amdgcn_wave_barrier();                                                                             \
        _Pragma("unroll") for (int k = 0; k < SROWS / 8; ++k) {                                                      \
          const int row_ = (le >> 3) + 8 * k, n0_ = 32 * (NPG * nb + pg) + sr + 8 * k;                               \
          const u32x4 o_ = *(const u32x4*)(stg + row_ * 128 + (((le & 7) ^ (row_ & 7)) * 16));                       \
          if (!RAGGED || n0_ + (le >> 3) < n_pos_)                                                                              \
            __builtin_nontemporal_store(o_, (u32x4*)(Ob_ + ((uint32_t)n0_ * (uint32_t)(DHHV * 2) + lofs_)));         \
        }                                                                                                            \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                       \
        __builtin_amdgcn_wave_barrier();                                                                             \
      }                                                                                                              \
    }                                                                                                                \
  }
    for (int rd = 0; rd < n_rounds; ++rd) {
      if (!win_decode(it, rd, vid, G, n_items, NWIN)) continue;
      const int bh = it.bh, c0 = 2 * it.win;
      const int n_pos = RAGGED ? S - 256 * it.win : 256;
      const float g01 = a.g.graw[(size_t)bh * NC + c0];
      const bool no_state = it.win == zero_win;

      // ================================================================================= phase S: the score blocks
      float dot = 0.f;
      {
        f32x16 sacc[5];
        auto s_step = [&](const unsigned char* slab) {
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
              mfma32<F16>(sacc[e], A, e < 3 ? Ba : Bc);  // rows: keys j, columns: positions t
            }
          }
        };
        // q_t . n before the second chunk (before the first it is zero), as phase O does it with a state: two threads per
        // position, 16 of the slab's 32 entries each, in the order of the fragments
        auto s_dot = [&](const unsigned char* slab, int w) __attribute__((always_inline)) {
          const int td = opaque(tid);
          const int t = td >> 1, part = td & 1;
          const float* const np = nvec + DHQK + 32 * w + 16 * part;
          const uint4 q0 = *(const uint4*)(slab + t * 64 + (((2 * part) ^ win_f64(t)) * 16));
          const uint4 q1 = *(const uint4*)(slab + t * 64 + (((2 * part + 1) ^ win_f64(t)) * 16));
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const uint4 qv = x == 0 ? make_uint4(q0.x, q0.y, q1.x, q1.y) : make_uint4(q0.z, q0.w, q1.z, q1.w);
            const float4 na = *(const float4*)(np + 4 * x), nb4 = *(const float4*)(np + 8 + 4 * x);
            dot += lo2<F16>(qv.x) * na.x + hi2<F16>(qv.x) * na.y + lo2<F16>(qv.y) * na.z + hi2<F16>(qv.y) * na.w;
            dot += lo2<F16>(qv.z) * nb4.x + hi2<F16>(qv.z) * nb4.y + lo2<F16>(qv.w) * nb4.z + hi2<F16>(qv.w) * nb4.w;
          }
        };
        const bool with_dot = !IS_DV && no_state && a.use_nrow && tid >= 256;
        // (the first step stands before the loop: the finished tile that leaves in it must not be live around the loop)
        __syncthreads();
        const unsigned char* const first_slab = next_slab();
        if (!MULTI && pending) WH_EPILOGUE
#pragma unroll
        for (int e = 0; e < 5; ++e)
#pragma unroll
          for (int i = 0; i < 16; ++i) sacc[e][i] = 0.f;
        if (with_dot) s_dot(first_slab, 0);
        s_step(first_slab);
        for (int w = 1; w < NS; ++w) {
          __syncthreads();
          const unsigned char* const slab = next_slab();
          if (with_dot) s_dot(slab, w);
          s_step(slab);
        }
        // ---- gating: P = scores * exp(u_t - w_j + G) / sqrt(DHQK) (* rho_t), zero above the diagonal; forward: fp32 row
        // sums over the keys of the own chunk (the vectors were written at least one barrier ago)
        {
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
#pragma unroll
          for (int e = 0; e < 5; ++e) {
            if (e < 3 + blk.nc) {
              const int tb = e < 3 ? blk.ta : blk.tc, jb = e < 3 ? blk.ja + e : blk.jc + e - 3;
              const bool same = (tb >= 4) == (jb >= 4);
              const float un = uvec[32 * tb + r] + (same ? 0.f : g01);
              const float lq = lqr[32 * tb + r];
              unsigned char* const pbk = smem_raw + kWinPOfs + (tb * (tb + 1) / 2 + jb) * 2048 + r * 64;
              const int fr = win_f64(r);
              float rsum = 0.f;
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
                  rsum += pv[q];
                }
                *(uint2*)(pbk + ((g4 ^ fr) * 16) + 8 * h) = make_uint2(pack2<F16>(pv[0], pv[1]), pack2<F16>(pv[2], pv[3]));
              }
              if (!IS_DV && same) {
                const float tot = rsum + __shfl_xor(rsum, 32);
                if (h == 0) rows[(jb & 3) * 256 + 32 * tb + r] = tot;
              }
            }
          }
        }
      }

      for (int cg = 0; cg < NG; ++cg) {
        // ================================================== phase O: Out^T = State^T Xn^T over the head dimension
        auto o_step = [&](const unsigned char* slab, int w) {
          const unsigned char* const Xn = slab + 16384;
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          if (!IS_DV && cg == 0 && a.use_nrow) {
            // q_t . n before the chunk of t, two threads per position, 16 of the slab's 32 entries each (rows in fragment order)
            const int td = opaque(tid);
            const int t = td >> 1, part = td & 1;
            const float* const np = nvec + (t >> 7) * DHQK + 32 * w + 16 * part;
#pragma unroll
            for (int x = 0; x < 2; ++x) {
              // unit 2 part + x holds entries 4x .. 4x + 3 and 8 + 4x .. 8 + 4x + 3 of the sixteen
              const uint4 qv = *(const uint4*)(Xn + t * 64 + (((2 * part + x) ^ win_f64(t)) * 16));
              const float4 na = *(const float4*)(np + 4 * x), nb4 = *(const float4*)(np + 8 + 4 * x);
              dot += lo2<F16>(qv.x) * na.x + hi2<F16>(qv.x) * na.y + lo2<F16>(qv.y) * na.z + hi2<F16>(qv.y) * na.w;
              dot += lo2<F16>(qv.z) * nb4.x + hi2<F16>(qv.z) * nb4.y + lo2<F16>(qv.w) * nb4.z + hi2<F16>(qv.w) * nb4.w;
            }
          }
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            Frag A[2], B[NNB];
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) A[mb].u = *(const uint4*)(slab + ((2 * ci + mb) * 2 + ks) * 1024 + le * 16);
#pragma unroll
            for (int nb = 0; nb < NNB; ++nb) {
              const int row = 32 * (NPG * nb + pg) + r;
              B[nb].u = *(const uint4*)(Xn + row * 64 + (((2 * ks + h) ^ win_f64(row)) * 16));
            }
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int nb = 0; nb < NNB; ++nb) mfma32<F16>(acc[mb][nb], A[mb], B[nb]);
          }
        };
        auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int nb = 0; nb < NNB; ++nb)
#pragma unroll
              for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.f;
        };
        if constexpr (MULTI && CW == 64) {
          // (the first step in front of the loop, whose accumulators are cleared behind its barrier: with groups of 64 columns 2 to 3 %
          // of H -- 256/320, 32 heads of 400 positions 48.2 -> 46.6 us, 512/448, 16 heads 94.7 -> 93.0 -- with wider ones spills)
          if (!no_state) {
            __syncthreads();
            const unsigned char* const slab = next_slab();
            clear();
            o_step(slab, 0);
            for (int w = 1; w < NS; ++w) {
              __syncthreads();
              o_step(next_slab(), w);
            }
          } else {
            clear();
          }
        } else {
          clear();
          const int ns = no_state ? 0 : NS;
          for (int w = 0; w < ns; ++w) {
            __syncthreads();
            o_step(next_slab(), w);
          }
        }
        // ---- denominators (the row sums were written before the barrier passed last)
        auto denominators = [&]() __attribute__((always_inline)) {
          const int td = opaque(tid);
          const int t = td >> 1;
          dot += __shfl_xor(dot, 1);
          if ((td & 1) == 0) {
            float nmax = 1.f, iv = 1.f;
            const float mc = mcv[t];
            if (a.use_nrow) {
              float den = cs0v[t] * dot;
              const int kb = (t >> 5) & 3;
#pragma unroll
              for (int b4 = 0; b4 < 4; ++b4) den += b4 <= kb ? rows[b4 * 256 + t] : 0.f;
              const float floor_v = a.sig_gate ? 1.f : __expf(-mc);
              nmax = fmaxf(fabsf(den), floor_v);
              iv = 1.f / (nmax + a.eps);
            }
            inv[t] = iv;
            if (!RAGGED || c0 * kChunk + t < (int)Sp) a.nrow_out[(size_t)bh * Sp + (size_t)c0 * kChunk + t] = nmax;
            if (t < n_pos) {
              const size_t tg = (size_t)bh * S + (size_t)c0 * kChunk + t;
              if (a.n_out != nullptr) a.n_out[tg] = nmax;
              if (a.m_out != nullptr) a.m_out[tg] = mc;
            }
          }
        };
        if (!IS_DV && cg == 0 && !no_state) denominators();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < NNB; ++nb) {
          const float cs = csv[32 * (NPG * nb + pg) + (opaque(lane) & 31)];
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) acc[mb][nb] *= cs;
        }
        __builtin_amdgcn_sched_barrier(0);

        // ================================================== phase V: Out^T += Xw^T P over the positions of the window
#pragma unroll
        for (int z = 0; z < NVS; ++z) {
          __syncthreads();
          const unsigned char* const Zs = next_slab();
          if (!IS_DV && z == 0 && cg == 0 && no_state) denominators();
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
          const int q16 = (le >> 4) & 1, i16 = le & 15;
          const int krow = 8 * h + (i16 >> 2);
          const int zun = 2 * q16 + ((i16 & 3) >> 1), zin = 8 * (i16 & 1);
#pragma unroll
          for (int zh = 0; zh < VROWS / 32; ++zh) {
            const int ob = z * (VROWS / 32) + zh;  // 32-position block of the contraction index
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
              Frag A[2];
#pragma unroll
              for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                  const int row = 32 * zh + 16 * kk + krow + 4 * half;
                  const int un = 8 * ci + 4 * mb + zun;
                  A[mb].d[half] = lds_read_tr16(Zs + row * (CW * 2) + ((un ^ win_zsw<CW * 2>(row)) * 16) + zin);
                }
#pragma unroll
              for (int nb = 0; nb < NNB; ++nb) {
                const WinSide side = win_side(IS_DV, ob, nb, NPG);
                if (side == kWinOff) continue;
                const int nbk = NPG * nb + pg;
                const bool live = side == kWinOn || (IS_DV ? ob >= nbk : ob <= nbk);
                // (the matrix instructions stay unconditional: accumulators that pass through a branch get copied)
                Frag Ax[2], B;
                B.u = Ax[0].u = Ax[1].u = make_uint4(0u, 0u, 0u, 0u);
                if (live) {
                  Ax[0] = A[0];
                  Ax[1] = A[1];
                  if (IS_DV) {
                    const unsigned char* const pbk = smem_raw + kWinPOfs + (ob * (ob + 1) / 2 + nbk) * 2048;
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                      const int row = 16 * kk + krow + 4 * half;
                      B.d[half] = lds_read_tr16(pbk + row * 64 + ((zun ^ win_f64(row)) * 16) + zin);
                    }
                  } else {
                    const unsigned char* const pbk = smem_raw + kWinPOfs + (nbk * (nbk + 1) / 2 + ob) * 2048;
                    B.u = *(const uint4*)(pbk + r * 64 + (((2 * kk + h) ^ win_f64(r)) * 16));
                  }
                }
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) mfma32<F16>(acc[mb][nb], Ax[mb], B);
              }
            }
          }
        }
        if constexpr (NORM) {
          // ---- sums over this wave's 64 columns of every row, from the finished accumulators
          const int le = opaque(lane);
          const int r = le & 31, h = le >> 5;
#pragma unroll
          for (int nb = 0; nb < NNB; ++nb) {
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const float x = acc[mb][nb][i];
                s1 += x;
                s2 = __builtin_fmaf(x, x, s2);
              }
            s1 += __shfl_xor(s1, 32);
            s2 += __shfl_xor(s2, 32);
            if (h == 0) {
              nst[ci * 512 + 32 * (NPG * nb + pg) + r] = s1;
              nst[ci * 512 + 256 + 32 * (NPG * nb + pg) + r] = s2;
            }
          }
        }
        pending = true;
        prev = it;
        prev_cg = cg;
        if constexpr (MULTI) WH_EPILOGUE
      }
    }
    if (pending) {  // (a workgroup without a window passes no barrier at all, like its producers)
      __syncthreads();
      if constexpr (!MULTI) WH_EPILOGUE
    }
#undef WH_EPILOGUE
  }
}

namespace {
template <int CW, bool MULTI, bool IS_DV, bool NORM, bool RAGGED, bool F16>
const char* launch_window_hv_r(const ParHvArgs& a, int BH, hipStream_t stream) {
  const long long n_items = (long long)BH * ((a.NC + 1) / 2);
  if (n_items >= (1ll << 31)) return "window_hv: too many work items";
  if ((size_t)a.S * (size_t)(a.DHHV > a.DHQK ? a.DHHV : a.DHQK) * 2 >= ((size_t)1 << 32))
    return "window_hv: one (batch, head) slab of an input exceeds 4 GiB";
  const int cus = device_cu_count();
  if (cus <= 0) return "window_hv: cannot read the number of compute units";
  int G = (int)(n_items < cus ? n_items : cus);
  if (n_items > G && G >= 8) G -= G % 8;  // (fewer items than CUs: one each, two rounds otherwise)
  const int n_rounds = (int)((n_items + G - 1) / G);
  static LdsLimit lds;
  if (!lds.allow((const void*)window_hv_kernel<CW, MULTI, IS_DV, NORM, RAGGED, F16>, kHvSmem))
    return "window_hv: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((window_hv_kernel<CW, MULTI, IS_DV, NORM, RAGGED, F16>), dim3(G), dim3(768), kHvSmem, stream, a, (int)n_items, n_rounds);
  return nullptr;
}
template <int CW, bool MULTI, bool IS_DV, bool NORM>
const char* launch_window_hv_n(const ParHvArgs& a, int BH, hipStream_t stream) {
  if (a.S % (2 * kChunk) != 0)
    return a.f16 ? launch_window_hv_r<CW, MULTI, IS_DV, NORM, true, true>(a, BH, stream)
                 : launch_window_hv_r<CW, MULTI, IS_DV, NORM, true, false>(a, BH, stream);
  return a.f16 ? launch_window_hv_r<CW, MULTI, IS_DV, NORM, false, true>(a, BH, stream)
               : launch_window_hv_r<CW, MULTI, IS_DV, NORM, false, false>(a, BH, stream);
}
template <int CW, bool MULTI>
const char* launch_window_hv_c(const ParHvArgs& a, int BH, bool is_dv, hipStream_t stream) {
  if (is_dv) return launch_window_hv_n<CW, MULTI, true, false>(a, BH, stream);
  if constexpr (!MULTI) {
    if (a.head_norm != 0) return launch_window_hv_n<CW, MULTI, false, true>(a, BH, stream);
  }
  return launch_window_hv_n<CW, MULTI, false, false>(a, BH, stream);
}
}  // namespace

// Where the window kernel is the faster one.  Its workgroups are one per CU and walk a window in 10 to 30 steps of one
// slab, so a launch of few windows leaves CUs idle that the tiled kernel (two workgroups per chunk of 128 positions, all
// value columns) fills: with groups of 256 columns the two meet at half a window per CU (H, us, window / tiled: 256/256 31 / 25
// at 64 windows, 32 / 34 at 128, 43 / 65 at 256).  With groups of 64 and 128 columns the window kernel wins from one window on
// (64/64: 14 / 27 at 8 windows, 17 / 55 at 256; 128/128 18 / 23, 23 / 49): the tiled kernel has one or two waves per workgroup
// there.  So it does with three groups of 64 (128/192: 26 / 33 at 8, 31 / 160 at 256); with five and more one workgroup's
// walk through the groups takes longer than the tiled kernel as long as that has a workgroup and a CU for every group of its
// own (128/384: 39 / 24 at 16 windows, 128/320 35 / 32 at 8, 256/640 76 / 30), and far less once it has not (128/384: 40 / 53
// at 64, 128/320 35 / 123 at 16).
bool window_hv_preferred(const ParHvArgs& a, int BH) {
  if (!window_hv_supported(a)) return false;
  if (a.DHHV % 256 == 0) return 2ll * BH * ((a.NC + 1) / 2) >= device_cu_count();
  return a.DHHV < 320 || !par_hv_group_each(a, BH);
}

bool window_hv_supported(const ParHvArgs& a) {
  const bool norm_ok = a.head_norm == 0 || a.DHHV == 64 || a.DHHV == 128 || a.DHHV == 256;  // complete rows in one group
  return a.stride == 2 && a.DHQK % 64 == 0 && a.DHQK <= kHvMaxDhqk && a.DHHV % 64 == 0 && norm_ok;
}

const char* launch_window_hv(const ParHvArgs& a, int BH, bool is_dv, hipStream_t stream) {
  if (!window_hv_supported(a)) return "window_hv: unsupported shape (needs state stride 2, DHQK at most 512)";
  if (a.head_norm != 0 && (is_dv || a.norm_mean == nullptr || a.norm_rstd == nullptr))
    return "window_hv: the head norm belongs to the forward and needs its mean / rstd outputs";
  if (a.DHHV == 64) return launch_window_hv_c<64, false>(a, BH, is_dv, stream);
  if (a.DHHV == 128) return launch_window_hv_c<128, false>(a, BH, is_dv, stream);
  if (a.DHHV == 256) return launch_window_hv_c<256, false>(a, BH, is_dv, stream);
  if (a.DHHV % 256 == 0) return launch_window_hv_c<256, true>(a, BH, is_dv, stream);
  return launch_window_hv_c<64, true>(a, BH, is_dv, stream);
}

}  // namespace mlstm
