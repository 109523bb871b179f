// What the two window kernels (window_hv.hip, window_qk.hip) share: a WINDOW is the pair of chunks (256 positions) that
// share a kept state at state stride 2; its causal score matrix is a lower triangle of 8 x 8 blocks of 32 x 32, 36
// blocks, which eight consumer waves compute together and keep in LDS as 16-bit values.
#pragma once
#include "common.h"

namespace mlstm {

struct WinItem {
  int bh, win;  // (batch * head), window
};

// Work item of workgroup `vid` in round `round`: consecutive workgroups take consecutive windows (neighbours share rows
// through the L2 of their XCD); the assignment rotates by one per round.
__device__ __forceinline__ bool win_decode(WinItem& it, int round, int vid, int G, int n_items, int NWIN) {
  const int rot = (vid + round) % G;
  const long long idx = (long long)round * G + rot;
  if (idx >= n_items) return false;
  it.win = (int)idx % NWIN;
  it.bh = (int)idx / NWIN;
  return true;
}

constexpr float kWinLog2e = 1.4426950408889634f;
constexpr int kWinSlot = 32768;          // bytes per ring slot (the largest slab)
constexpr int kWinPOfs = 2 * kWinSlot;   // P behind the two slots: 36 blocks of 32 x 32 (2 KB each, 64-byte rows, swizzled)
constexpr int kWinPBytes = 36 * 2048;

// Swizzles of 16-byte units.  LDS has 64 banks of 4 bytes and serves a 16-byte read in groups of 16 lanes, 0-3 12-15 20-27 and
// 4-11 16-19 28-31 (and the same of lanes 32-63), an 8-byte one, transposing or not, in groups of 32.
// Tiles with 64-byte rows (operand rows of 32 columns, blocks of P), four rows to a line of banks: of 32 rows read at one unit a group
// has four of every residue mod 4, whose numbers / 4 differ mod 4; the 4 rows x 4 units patch of a transposing read is a line.
__device__ __forceinline__ int win_f64(int row) { return (row >> 2) & 3; }
// Tiles with rows of RB = 128, 256 or 512 bytes: a transposing read takes 4 neighbouring units of 4 consecutive rows, and a read of 8
// bytes of one unit 32 rows.  (512: 8 rows further on, which is where the next piece of a thread goes, it is the same again.)
// Against swizzles for groups of 8 and 16 neighbouring lanes, which two lanes of every group shared a bank with (us, before / after):
// dQ / dK of 256/512, 32 heads of 16384 759 / 747, 128 of 1024 188 / 185; conflicts 0.40 / 0.12 of the LDS cycles.  Rows of 128 bytes
// keep theirs, with which the patch falls on distinct banks too: one that also spreads the 8-byte reads measured slower, for a reason not
// found (forward and backward, with that / this: 64/64, 24 heads of 9984 239 / 235, 32 of 4096 148 / 145; 128/256, 32 of 8192 546 / 539).
template <int RB>
__device__ __forceinline__ int win_zsw(int row) {
  if (RB == 128) return 2 * (row & 3);
  return ((row & 3) << 2) | (RB == 256 ? (row >> 2) & 3 : ((row >> 2) & 1) << 1);
}

// The blocks (tb, jb) of the lower triangle that a consumer wave computes: three blocks of row ta (keys ja, ja + 1, ja + 2)
// and up to two of row tc (keys jc, jc + 1).  With at most two rows per wave and the split between them fixed, the
// operand of a row is read once for all its blocks: seven fragments feed five matrix instructions instead of ten.
// A wave computes a missing fifth (fourth) block all the same and drops it (nc = how many of the last two count).
struct WinBlocks {
  int ta, ja, tc, jc, nc;
};
__device__ __forceinline__ WinBlocks win_blocks(int wave) {
  switch (wave) {
    case 0: return {7, 0, 7, 6, 2};
    case 1: return {7, 3, 6, 3, 2};
    case 2: return {6, 0, 6, 5, 2};
    case 3: return {5, 0, 4, 3, 2};
    case 4: return {5, 3, 1, 0, 2};
    case 5: return {4, 0, 3, 3, 1};
    case 6: return {3, 0, 0, 0, 1};
    default: return {2, 0, 2, 1, 0};
  }
}

// Which blocks of P a wave multiplies: those of its position blocks NPG * nb + pg (pg < NPG) that lie on the causal side of
// the contraction block ob (ahead: contraction over later positions).  Known at compile time except for which waves have it.
// A block on the other side is left out, operands and all: P holds nothing there, and as an operand of zeros it would turn a
// NaN or infinity in the rows of block ob into NaN at every position of the window (now: at those of its own 32 at most).
// Without their matrix instructions and with the loop over the blocks unrolled (us, before / after): H at 128/256 with 262144
// token-heads 116 / 114, dQ / dK at 256/256 with 131072 135 / 130, at 512/1024 with 32768 199 / 192, at 256/512 with 64 heads of
// 1000 98 / 94; dV and the small tiles the same.
enum WinSide { kWinOff, kWinSome, kWinOn };
constexpr WinSide win_side(bool ahead, int ob, int nb, int NPG) {
  const int lo = NPG * nb, hi = lo + NPG - 1;
  if (ahead) return ob >= hi ? kWinOn : (ob < lo ? kWinOff : kWinSome);
  return ob <= lo ? kWinOn : (ob > hi ? kWinOff : kWinSome);
}

}  // namespace mlstm
