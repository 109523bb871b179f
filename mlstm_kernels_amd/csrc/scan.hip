// Inter-chunk state scan of the chunkwise mLSTM, forward (C states) and backward (dC states).
//
//   forward :  C_c  = gbar_c * C_{c-1} + K_c^T (abar . V_c)          c = 0 .. NC-1      (and n likewise)
//   backward:  dC_{c-1} = gbar_c * dC_c + Q_c^T (rho . dH_c)          c = NC-1 .. 0,
//              rho_t = bbar_t / sqrt(DHQK) / (nrow_t + eps)
//
// (mlstm_kernels/torch/chunkwise/native/fw.py:88-121 and bw.py:67-98 in the reference.)  Both are the same
// kernel: a (DHQK x DHHV) fp32 state tile stays in MFMA accumulators for the whole sequence; per chunk the
// tile is first written out as bf16 operand fragments (the state *before* the update, which is what the
// chunk-parallel kernels consume), then decayed and updated with X_c^T (rowscale . Y_c), contraction over
// the 128 chunk positions.  Both operands have the contraction index as their slow memory dimension, so
// both are staged row-major in LDS and fetched with the transposing 64-bit LDS read.
//
// The row scale is applied to Y (the narrower operand of the tile) in fp32 before rounding to bf16.  For the
// forward the scaled rows are split into a bf16 head and a bf16 remainder (two MFMAs) so that the final
// state keeps ~16 mantissa bits: a single bf16 rounding of abar*V leaves a relative error of about 1.5e-3
// in C, above the 1e-3 the state is specified to.
//
// Two kernels: scan_roles_kernel (below, second) -- every scan -- and scan_kernel with the head + remainder split for
// forwards that return the last state and in which many chunks still weigh in it (it continues where the first one
// stopped; the state passes through the caller's last-state buffers).  Where only a few do, scan_roles_kernel runs those
// chunks twice, once with the heads and once with the remainders.  Same tiling, same arithmetic, same results.
//
// A scan of few (batch, head) pairs has too few state tiles to fill the chip and walks the sequence chunk by chunk at
// 1.6 to 1.9 us, whatever the memory could deliver.  It is cut into segments of the sequence that run side by side: a first
// launch accumulates every segment but the last from zero, a second one runs all segments from the state before them,
// which is the decayed sum of the first launch's results (the decay factors depend on the gates only).
//
// Workgroups are renumbered so that all tiles of one (batch, head) run on the same XCD (the hardware deals
// consecutive workgroup ids round-robin to the 8 XCDs): the K/V rows every tile of a head re-reads then hit
// that XCD's L2 instead of going to HBM once per tile.
#include "common.h"
#include "kernels.h"

namespace mlstm {

constexpr int kGBlock = 256;  // chunks per refill of the decay-factor table in LDS

// A chunk is staged in 128 / PS pieces of PS positions (the contraction over positions is a plain sum): the
// smaller the piece, the smaller the LDS tiles and the prefetch registers, but the more barriers per chunk.
// scan_kernel: eight waves per 128 x 128 tile (64 x 32 per wave), one workgroup per CU.  scan_roles_kernel: two LDS
// buffers and sixteen waves in two roles -- eight producer waves fetch, scale and stage the rows of chunk c+1 while
// eight consumer waves do the fragment reads and matrix instructions of chunk c (one barrier per chunk); the
// normaliser recurrence rides as three more operand columns on the consumers' matrix pipe.
// What pays is more instruction streams per SIMD inside the same workgroup: the phases of a chunk (staging, state
// emission, matrix work) are serial per wave; two waves per SIMD overlap one's LDS and conversion latencies with the
// other's matrix instructions, and four waves in two roles keep the conversion arithmetic and the matrix
// instructions in different waves altogether.
// The remainder of the value operand serves the last state only, and chunk c enters the last state with the weight
// W_c = product of the decay factors of the chunks after it (<= 1, non-increasing towards the start).  Chunks whose
// weight is below 2^-8 are accumulated without the remainder: their rounding (2^-9 relative) then reaches the last
// state at 2^-17 of its scale.  Returns the first chunk that carries the remainder (at most NC - 1); every wave
// computes it for itself, and every kernel that needs it gets the same value.
__device__ __forceinline__ int first_remainder_chunk(const float* gbar_bh, int NC, int lane) {
  float carry = 1.f;
  int cnt = 0;
  for (int base = 0; base < NC; base += kWave) {
    const int cc = NC - 1 - (base + lane);                       // walking from the last chunk towards the first
    const float gv = cc >= 0 ? gbar_bh[cc] : 0.f;
    float incl = gv;                                            // inclusive prefix product over the lanes
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const float up = __shfl_up(incl, o);
      if (lane >= o) incl *= up;
    }
    float excl = __shfl_up(incl, 1);
    if (lane == 0) excl = 1.f;
    const bool need = cc >= 0 && carry * excl >= 0.00390625f;    // W_cc >= 2^-8
    const int n_need = __popcll(__ballot(need));
    cnt += n_need;
    if (n_need < kWave) break;                                   // weights only fall from here on
    carry *= __shfl(incl, kWave - 1);
  }
  return __builtin_amdgcn_readfirstlane(NC - cnt);
}

// Whether the chunks that carry the remainder run twice in scan_roles_kernel (once with the 16-bit heads, once with the
// remainders) or go to scan_kernel in a launch of its own.  A second run costs a chunk's time again (2.3 us at B = 4,
// S = 16384, against 3.6 us for both operands at once in scan_kernel), the launch and its tail a fixed 12 us per round
// of workgroups.  repeat_all: they always do (launch_scan has the rule); otherwise where they are at most a quarter of all.
__device__ __forceinline__ bool scan_repeats_late(const ScanArgs& a, int c_lo) { return a.repeat_all || 4 * (a.NC - c_lo) <= a.NC; }

#define SCAN_WPE(HILO_, WCOLS_) ((WCOLS_) == 64 && (HILO_) ? 1 : 2)
// WCOLS = value columns per wave (64 or 32): with 32 a 128 x 128 tile takes eight waves, two per SIMD, each with
// half the staging work and half the accumulators.
template <bool V>
struct BoolTag {
  static constexpr bool value = V;
};

template <int RT, int WT, bool HILO, int PS, int WCOLS, bool F16>
__global__ __launch_bounds__(64 * (RT / 64) * (WT / WCOLS))
    __attribute__((amdgpu_waves_per_eu(SCAN_WPE(HILO, WCOLS), SCAN_WPE(HILO, WCOLS)))) void scan_kernel(ScanArgs a) {
  constexpr int WC = WT / WCOLS;
  constexpr int NBW = WCOLS / 32;  // 32-column accumulator blocks per wave
  constexpr int NT = 64 * (RT / 64) * WC;
  constexpr int XS = RT + 32;  // LDS row strides (elements): consecutive rows start 16 banks (64 bytes) apart
  constexpr int YS = WT + 32;
  constexpr int XV = PS * RT / 8 / NT;   // 16-byte vectors per thread per piece
  constexpr int YV = PS * WT / 8 / NT;
  constexpr int NP = kChunk / PS;        // pieces per chunk
  constexpr int XROWS = NT / (RT / 8);   // rows covered by one sweep of the workgroup over X
  // The n update is summed in one order whatever the tile's width, so that the width changes no bit: rows j, j + 32, ... first,
  // then the sums of j and j + 16, then those.  A sweep covers 32 rows (a wave's two sums meet behind LDS) or 16 (in front).
  constexpr int NSET = 32 / XROWS;
  static_assert(XV >= 1 && YV >= 1 && PS % 16 == 0, "piece too small for this tile");
  static_assert((XROWS == 32 || XROWS == 16) && XV % NSET == 0, "the sums of n");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  uint16_t* Xs = (uint16_t*)smem_raw;
  uint16_t* Yh = Xs + PS * XS;
  uint16_t* Yl = Yh + PS * YS;
  float* npart = (float*)(Yl + (HILO ? PS * YS : 0));  // [XROWS][RT] partial sums of the n update
  float* gl = npart + XROWS * RT;                       // [kGBlock] decay factors of the next chunks, in scan order
  float* scl = gl + kGBlock;                            // [2][128] row scales of the chunk being staged / the next one

  // the wave index is made scalar so that branches on it are scalar branches (accumulators stay in place)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WC, wc = wave % WC;
  const int r = lane & 31, h = lane >> 5;
  // ---- XCD-aware renumbering: linear id -> (xcd, slot) -> contiguous range of ids per XCD
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  {
    const int total = gridDim.x * gridDim.y * gridDim.z;
    if (total % 8 == 0) {
      const int lin = bx + gridDim.x * (by + gridDim.y * bz);
      const int virt = (lin % 8) * (total / 8) + lin / 8;
      bx = virt % gridDim.x;
      by = (virt / gridDim.x) % gridDim.y;
      bz = virt / (gridDim.x * gridDim.y);
    }
  }
  const int bh = bz;
  const int d_tile = bx * RT, w_tile = by * WT;
  const int d_wave = d_tile + wr * 64, w_wave = w_tile + wc * WCOLS;
  const int DHQK = a.DHQK, DHHV = a.DHHV, S = a.S, NC = a.NC;
  const size_t Sp = (size_t)NC * kChunk;
  // c_lo = first chunk that carries the remainder of the value operand
  int c_lo = 0;
  if constexpr (HILO) {
    if (!a.backward) c_lo = a.all_remainder ? 0 : first_remainder_chunk(a.gbar + (size_t)bh * NC, NC, lane);
    if (a.part == 2 && scan_repeats_late(a, c_lo)) return;  // the first launch ran everything
  }

  f32x16 acc[2][NBW];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int wb = 0; wb < NBW; ++wb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float v0 = 0.f;
        const float* init = a.part == 2 ? a.final_out : a.init;  // part 2 continues from the first launch's state
        if (init != nullptr) {
          const int d = d_wave + 32 * db + 8 * (i / 4) + 4 * h + (i % 4);
          const int w = w_wave + 32 * wb + r;
          v0 = init[((size_t)bh * DHQK + d) * DHHV + w];
        }
        acc[db][wb][i] = v0;
      }
    }
  const bool do_n = (a.nstates != nullptr) && by == 0;
  float nval = 0.f;
  {
    const float* n_init = a.part == 2 ? a.n_final : a.n_init;
    if (do_n && tid < RT && n_init != nullptr) nval = n_init[(size_t)bh * DHQK + d_tile + tid];
  }

  const uint16_t* Xg = a.X + (size_t)bh * S * DHQK + d_tile;
  const uint16_t* Yg = a.Y + (size_t)bh * S * DHHV + w_tile;

  uint4 xr[XV], yr[YV];
  // Row scales (forward: abar_j; backward: bbar_t / sqrt(DHQK) / (nrow_t + eps)) go through a table in LDS instead of
  // one 4-byte load per staged vector: every thread fetches the factor of ONE row two chunks ahead (a single load
  // instruction per wave and chunk), the table entry is written while the chunk before it is staged.  The vector
  // memory path of the CU (64 bytes per clock for loads, stores and their address processing) is what the scan
  // queues on, so its instruction count matters.
  const int srow = tid & (kChunk - 1);
  const float* const nrow_or_dummy = a.nrow != nullptr ? a.nrow : a.scale_a;
  float s_raw = 0.f, s_nrm = 1.f;
  auto load_scales = [&](int c) {
    const int cc = min(max(c, 0), NC - 1);
    const int t = cc * kChunk + srow;
    s_raw = a.scale_a[bh * Sp + t];
    s_nrm = nrow_or_dummy[bh * Sp + t];
  };
  // The prefetch only LOADS: any arithmetic on a loaded value here would make the wave wait for the whole batch of
  // loads before it starts the matrix work they are meant to overlap with.
  auto prefetch = [&](int c, int piece) {
#pragma unroll
    for (int v = 0; v < XV; ++v) {
      const int idx = tid + v * NT;
      const int j = idx / (RT / 8), cv = idx % (RT / 8);
      const int t = c * kChunk + piece * PS + j;
      xr[v] = t < S ? *(const uint4*)(Xg + (size_t)t * DHQK + cv * 8) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < YV; ++v) {
      const int idx = tid + v * NT;
      const int j = idx / (WT / 8), cv = idx % (WT / 8);
      const int t = c * kChunk + piece * PS + j;
      yr[v] = t < S ? *(const uint4*)(Yg + (size_t)t * DHHV + cv * 8) : make_uint4(0, 0, 0, 0);
    }
  };

  const int c_first_all = a.backward ? NC - 1 : 0, c_step = a.backward ? -1 : 1;
  // part 2 of a forward scan in two launches: the chunks from c_lo on, continuing from the state the first launch left
  // in final_out / n_final (loaded above)
  const int c_first = a.part == 2 ? c_lo : c_first_all;
  const int NCR = a.part == 2 ? NC - c_lo : NC;  // chunks this launch runs
  // row scales of the first chunk straight into the table, those of the second chunk into the prefetch register
  {
    const int t = c_first * kChunk + srow;
    float sc0 = t < S ? a.scale_a[bh * Sp + t] : 0.f;
    if (a.backward) {
      sc0 *= a.qk_scale;
      if (a.nrow != nullptr) sc0 /= (a.nrow[bh * Sp + t] + a.eps);
    }
    if (tid < kChunk) scl[srow] = sc0;
  }
  load_scales(NCR > 1 ? c_first + c_step : c_first);
  prefetch(c_first, 0);
  for (int hit = 0; hit < NCR * NP; ++hit) {
    const int it = hit / NP, piece = hit % NP;
    const int c = c_first + it * c_step;
    // The decay factors come from LDS, a block of chunks at a time: read straight from global memory inside the
    // loop, the factor would sit behind the prefetch of the next chunk (loads complete in order) and the matrix
    // work would wait for the whole prefetch in every iteration.
    if (piece == 0 && (it & (kGBlock - 1)) == 0) {
      __syncthreads();
      for (int k = tid; k < kGBlock && it + k < NCR; k += NT) gl[k] = a.gbar[(size_t)bh * NC + c + k * c_step];
      // visible after the barrier that follows the staging below
    }
    // ---- registers -> LDS (Y rows scaled in fp32, then rounded / split); partial sums of sum_j abar_j k_j
    const float* scur = scl + (it & 1) * kChunk + piece * PS;  // written while the previous chunk was staged
    const bool with_lo = HILO && c >= c_lo;                    // uniform over the workgroup
    if (piece == 0 && tid < kChunk) {
      // the next chunk's row scales (fetched two chunks ahead) into the other half of the table
      const int t = (c + c_step) * kChunk + srow;
      float sn = (it + 1 < NCR && t < S) ? s_raw : 0.f;
      if (a.backward) {
        sn *= a.qk_scale;
        if (a.nrow != nullptr) sn /= (s_nrm + a.eps);
      }
      scl[((it + 1) & 1) * kChunk + srow] = sn;
    }
    float np[NSET][8] = {};
#pragma unroll
    for (int v = 0; v < XV; ++v) {
      const int idx = tid + v * NT;
      const int j = idx / (RT / 8), cv = idx % (RT / 8);
      *(uint4*)(Xs + j * XS + cv * 8) = xr[v];
      if (do_n) {
        const uint32_t in[4] = {xr[v].x, xr[v].y, xr[v].z, xr[v].w};
        const float xsc = scur[j];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          np[v % NSET][2 * p] += xsc * lo2<F16>(in[p]);
          np[v % NSET][2 * p + 1] += xsc * hi2<F16>(in[p]);
        }
      }
    }
    if (do_n) {
      // thread (row group tid/(RT/8), column vector tid%(RT/8)) holds the sums over its XV rows
      if constexpr (NSET == 2) {
#pragma unroll
        for (int p = 0; p < 8; ++p) np[0][p] += np[1][p];
      }
      float* dst = npart + (tid / (RT / 8)) * RT + (tid % (RT / 8)) * 8;
      *(float4*)dst = make_float4(np[0][0], np[0][1], np[0][2], np[0][3]);
      *(float4*)(dst + 4) = make_float4(np[0][4], np[0][5], np[0][6], np[0][7]);
    }
#pragma unroll
    for (int v = 0; v < YV; ++v) {
      const int idx = tid + v * NT;
      const int j = idx / (WT / 8), cv = idx % (WT / 8);
      const uint32_t in[4] = {yr[v].x, yr[v].y, yr[v].z, yr[v].w};
      uint32_t hi[4], lo[4];
      const float sc = scur[j];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const float e0 = lo2<F16>(in[p]) * sc;
        const float e1 = hi2<F16>(in[p]) * sc;
        hi[p] = pack2<F16>(e0, e1);
        if (HILO) lo[p] = pack2<F16>(e0 - lo2<F16>(hi[p]), e1 - hi2<F16>(hi[p]));
      }
      *(uint4*)(Yh + j * YS + cv * 8) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      if (HILO) {
        if (with_lo) *(uint4*)(Yl + j * YS + cv * 8) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      }
    }
    __syncthreads();
    if (hit + 1 < NCR * NP) prefetch(piece + 1 < NP ? c : c + c_step, piece + 1 < NP ? piece + 1 : 0);
    if (piece == 0) load_scales(c + 2 * c_step);

    // ---- emit the state before this chunk's update as bf16 operand fragments, at the kept boundaries only: forward
    // the state before every stride-th chunk, backward the gradient of the state after the last chunk of every group
    // of `stride` chunks (and after the last chunk of the sequence); slot c / stride either way
    const bool keep = a.backward ? (c == NC - 1 || (c + 1) % a.stride == 0) : (c % a.stride == 0);
    if (piece == 0 && keep) {
      const size_t ND = DHQK / 16, NW = DHHV / 32;
      const size_t NCS = (size_t)(NC + a.stride - 1) / a.stride;
      uint4* st = (uint4*)a.states + ((size_t)bh * NCS + c / a.stride) * NW * ND * 64;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int wb = 0; wb < NBW; ++wb) {
          const size_t W32 = (w_wave + 32 * wb) / 32, D16 = (d_wave + 32 * db) / 16;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            uint4 f;
            f.x = pack2<F16>(acc[db][wb][8 * half + 0], acc[db][wb][8 * half + 1]);
            f.y = pack2<F16>(acc[db][wb][8 * half + 2], acc[db][wb][8 * half + 3]);
            f.z = pack2<F16>(acc[db][wb][8 * half + 4], acc[db][wb][8 * half + 5]);
            f.w = pack2<F16>(acc[db][wb][8 * half + 6], acc[db][wb][8 * half + 7]);
            // non-temporal: the fragments are read by a later kernel; kept out of the L2 they do not evict the K/V
            // rows the tiles of a head share
            const u32x4 fv = {f.x, f.y, f.z, f.w};
            __builtin_nontemporal_store(fv, (u32x4*)(st + (W32 * ND + D16 + half) * 64 + lane));
          }
        }
    }
    // ---- decay (once per chunk), then accumulate X^T (scale . Y) over the positions of this piece
    const float g = piece == 0 ? gl[it & (kGBlock - 1)] : 1.f;
    if (piece == 0) {
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int wb = 0; wb < NBW; ++wb) acc[db][wb] *= g;
    }

    const int q16 = (lane >> 4) & 1, i16 = lane & 15;
    const int krow = 8 * h + (i16 >> 2), ncol = 16 * q16 + 4 * (i16 & 3);
    // two copies of the loop (with and without the remainder) rather than a branch inside it: the accumulators stay
    // where they are either way
    auto multiply = [&](auto lo_tag) {
      constexpr bool LO = decltype(lo_tag)::value;
#pragma unroll
      for (int js = 0; js < PS / 16; ++js) {
        Frag A[2], Bh[NBW], Bl[NBW];
#pragma unroll
        for (int db = 0; db < 2; ++db) {
          const uint16_t* p = Xs + (16 * js + krow) * XS + (wr * 64 + 32 * db + ncol);
          A[db].d[0] = lds_read_tr16(p);
          A[db].d[1] = lds_read_tr16(p + 4 * XS);
        }
#pragma unroll
        for (int wb = 0; wb < NBW; ++wb) {
          const int o = (16 * js + krow) * YS + (wc * WCOLS + 32 * wb + ncol);
          Bh[wb].d[0] = lds_read_tr16(Yh + o);
          Bh[wb].d[1] = lds_read_tr16(Yh + o + 4 * YS);
          if (LO) {
            Bl[wb].d[0] = lds_read_tr16(Yl + o);
            Bl[wb].d[1] = lds_read_tr16(Yl + o + 4 * YS);
          }
        }
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int wb = 0; wb < NBW; ++wb) {
            mfma32<F16>(acc[db][wb], A[db], Bh[wb]);
            if (LO) mfma32<F16>(acc[db][wb], A[db], Bl[wb]);
          }
      }
    };
    if (with_lo) multiply(BoolTag<HILO>{});
    else multiply(BoolTag<false>{});
    // ---- normaliser vector (forward, first column tile only): n = gbar n + sum_j abar_j k_j
    if (do_n && tid < RT) {
      if (piece == 0) {
        // three partial vectors per chunk (the consumer adds them up): this kernel keeps the whole sum in the first
        float* dst = a.nstates + ((size_t)bh * NC + c) * 3 * DHQK + d_tile + tid;
        dst[0] = nval;
        dst[DHQK] = 0.f;
        dst[2 * DHQK] = 0.f;
      }
      float s = 0.f;
#pragma unroll
      for (int g2 = 0; g2 < 16; ++g2) s += NSET == 2 ? npart[g2 * RT + tid] : npart[g2 * RT + tid] + npart[(g2 + 16) * RT + tid];
      nval = g * nval + s;
    }
    __syncthreads();
  }
  if (a.final_out != nullptr) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int wb = 0; wb < NBW; ++wb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int d = d_wave + 32 * db + 8 * (i / 4) + 4 * h + (i % 4);
          const int w = w_wave + 32 * wb + r;
          a.final_out[((size_t)bh * DHQK + d) * DHHV + w] = acc[db][wb][i];
        }
  }
  if (do_n && tid < RT && a.n_final != nullptr) a.n_final[(size_t)bh * DHQK + d_tile + tid] = nval;
}

template <int RT, int WT, bool HILO, bool F16>
static const char* launch_scan_f(const ScanArgs& a, int BH, hipStream_t stream) {
  constexpr int WCOLS = 32;
  constexpr int NT = 64 * (RT / 64) * (WT / WCOLS);
  constexpr int XROWS = NT / (RT / 8);
  constexpr int PS = 128;
  const size_t smem = (size_t)PS * (RT + 32) * 2 + (size_t)PS * (WT + 32) * 2 * (HILO ? 2 : 1) +
                      (size_t)(XROWS * RT + kGBlock + 2 * kChunk) * 4;
  static LdsLimit lds;
  if (!lds.allow((const void*)scan_kernel<RT, WT, HILO, PS, WCOLS, F16>, smem))
    return "scan: cannot raise the dynamic LDS limit";
  dim3 grid(a.DHQK / RT, a.DHHV / WT, BH);
  hipLaunchKernelGGL((scan_kernel<RT, WT, HILO, PS, WCOLS, F16>), grid, dim3(NT), smem, stream, a);
  return nullptr;
}

template <int RT, int WT, bool HILO>
static const char* launch_scan_t(const ScanArgs& a, int BH, hipStream_t stream) {
  return a.f16 ? launch_scan_f<RT, WT, HILO, true>(a, BH, stream) : launch_scan_f<RT, WT, HILO, false>(a, BH, stream);
}

// ---------------------------------------------------------------------------------------------------------------
// scan_roles_kernel: software pipeline over whole chunks with two LDS buffers and, per producer wave, two register
// sets.  While chunk c is multiplied out of one buffer, the rows of chunk c+1 (fetched two chunks earlier) are scaled,
// rounded and written into the other buffer, and the rows of chunk c+3 are requested into the register set this
// frees: ONE barrier per chunk, a global load has two chunk periods to arrive.  The tiles are unpadded (two buffers
// of a 128 x 128 tile pair fill 128 KB) and XOR-swizzled in 16-byte units so that the four rows a transposing read
// touches per half wave fall into four different 64-byte bank groups.
namespace {
template <int U>  // 16-byte units per tile row
__device__ __forceinline__ int scan_swz(int row) {
  return U == 8 ? ((row >> 1) & 1) << 2 : (row & 3) << 2;
}
struct ScanTrOff {
  int lo, hi;
};
// per-lane element offsets of the two transposing reads of a fragment (rows k0 + 8h .. +3 and +4 .. +7 of the
// contraction index, columns col0 .. col0+31) in a tile with ROWLEN elements per row; k0 is a multiple of 16, so the
// swizzle of the rows does not depend on it
template <int ROWLEN>
__device__ __forceinline__ ScanTrOff scan_tr_offsets(int col0, int lane) {
  const int q16 = (lane >> 4) & 1, i16 = lane & 15, h = lane >> 5;
  const int krow = 8 * h + (i16 >> 2);
  const int col = col0 + 16 * q16 + 4 * (i16 & 3);
  const int unit = col >> 3, sub = col & 7;
  ScanTrOff o;
  o.lo = krow * ROWLEN + ((unit ^ scan_swz<ROWLEN / 8>(krow)) << 3) + sub;
  o.hi = (krow + 4) * ROWLEN + ((unit ^ scan_swz<ROWLEN / 8>(krow + 4)) << 3) + sub;
  return o;
}
template <int ROWLEN>
__device__ __forceinline__ Frag scan_tr_frag(const uint16_t* tile, int k0, const ScanTrOff& o) {
  Frag f;
  f.d[0] = lds_read_tr16(tile + k0 * ROWLEN + o.lo);
  f.d[1] = lds_read_tr16(tile + k0 * ROWLEN + o.hi);
  return f;
}
}  // namespace

// What a workgroup of scan_roles_kernel runs of one job: chunks it_lo .. it_hi - 1 in scan order (forward: the chunk index,
// backward counted from the end), those from it_rep on twice in a row (heads, then remainders of the value rows).  Everything
// below is counted in runs p = 0 .. total - 1.  REP = false: nothing runs twice (no last state returned).
template <bool REP>
struct ScanRuns {
  int it_lo, it_rep, total;
  __device__ __forceinline__ void set(int lo, int hi, int rep) {
    it_lo = lo;
    it_rep = rep;
    total = hi - lo + (REP ? hi - rep : 0);
  }
  __device__ __forceinline__ int it(int p) const {  // scan index of run p
    const int q = p - (it_rep - it_lo);
    return !REP || q < 0 ? it_lo + p : it_rep + (q >> 1);
  }
  __device__ __forceinline__ bool rest(int p) const {  // whether run p is the second run of its chunk
    const int q = p - (it_rep - it_lo);
    return REP && q >= 0 && (q & 1);
  }
  __device__ __forceinline__ bool last(int p) const {  // whether run p is the last one of its chunk
    const int q = p - (it_rep - it_lo);
    return !REP || q < 0 || (q & 1);
  }
};

// One job of scan_roles_kernel: a state tile of one (batch, head), of one segment of the sequence.  The jobs of a workgroup
// are worked out once, at its start, and lie in LDS: worked out where they are needed, their divisions and their prefix
// products would stand five times in the producers' loop and cost it its scalar registers.
constexpr int kScanRounds = 32;  // jobs of a workgroup at most
struct ScanJob {
  int bh, seg, bx, by;
  int it_lo, it_hi, it_rep;  // see ScanRuns
  int end;                   // bit 0: the state after this job is the last one; bits 1..: 1 + scan index of the chunk in front
};                           // of which the state is wanted although the chunk is not run, or 0

// Job of workgroup `vid` in round `round`.  Consecutive workgroups of an XCD take consecutive jobs: all tiles of one (batch,
// head), which share its K / V rows in the L2.  The assignment rotates by one column of tiles per round, so that the first
// column's tiles, which carry n and may run a chunk more, do not all fall to the same workgroups.  A last round with jobs for some
// of the workgroups only gives every XCD an eighth of them: as they come they would all lie on the first ones (576 tiles of 64 x 64,
// 2048 positions, 54.9 -> 51.9 us without the last state).
template <int RT, int WT, bool REP, bool SEG>
__device__ __forceinline__ ScanJob scan_decode(const ScanArgs& a, int round, int vid, int lane) {
  ScanJob job = {0, 0, 0, 0, 0, 0, 0, 0};
  const int G = (int)gridDim.x, nx = a.DHQK / RT, ny = a.DHHV / WT;
  const long long left = a.n_jobs - (long long)round * G;  // jobs of this round and the later ones
  long long idx = (long long)round * G;
  if (left < G && G % 8 == 0) {
    // the last round, with jobs for some of the workgroups only: an eighth of them for each XCD
    const int per = G / 8, x = vid / per, l = (int)((vid % per + (unsigned)round * nx) % (unsigned)per);
    const int lo = x * (int)left / 8, hi = (x + 1) * (int)left / 8;
    if (l >= hi - lo) return job;
    idx += lo + l;
  } else {
    idx += (vid + (unsigned)round * nx) % (unsigned)G;
    if (idx >= a.n_jobs) return job;
  }
  job.bx = (int)idx % nx;
  job.by = ((int)idx / nx) % ny;
  const int z = (int)idx / (nx * ny);
  const int nrun = !SEG ? 1 : (a.seg_phase == 1 ? a.nseg - 1 : a.nseg);  // segments this launch runs
  job.bh = SEG ? z / nrun : z;
  job.seg = SEG ? z % nrun : 0;
  // chunks of the whole sequence that this tile runs; forward that returns the last state: the chunks from c_lo on carry the
  // remainder of the value operand and either run twice here or are left to scan_kernel (the state reached before them is
  // then handed over in final_out / n_final)
  int n_all = a.nstates != nullptr && job.by == 0 ? a.end_n : a.end_c, c_lo = a.NC;
  if (REP) {
    c_lo = a.all_remainder ? 0 : first_remainder_chunk(a.gbar + (size_t)job.bh * a.NC, a.NC, lane);
    if (!scan_repeats_late(a, c_lo)) n_all = c_lo;
  }
  job.it_lo = SEG ? job.seg * a.seg_len : 0;
  job.it_hi = max(SEG ? min(job.it_lo + a.seg_len, n_all) : n_all, job.it_lo);
  job.it_rep = max(min(c_lo, job.it_hi), job.it_lo);
  const bool is_end = !SEG || (n_all == 0 ? job.seg == 0 : (job.it_lo < n_all && job.it_lo + a.seg_len >= n_all));
  const bool emit = !REP && n_all < a.NC && (!SEG || (a.seg_phase == 2 && job.it_lo <= n_all && n_all < job.it_lo + a.seg_len));
  job.end = (is_end ? 1 : 0) | (emit ? (n_all + 1) << 1 : 0);
  return job;
}

// Segment states between the two launches of a segmented scan, in the register order of the consumer waves:
// [(batch * head * (segments - 1) + segment)][tile][consumer wave][8][64 lanes][4], behind them n [..][DHQK].
struct ScanSeg {
  float* c;
  float* n;
};
__device__ __forceinline__ ScanSeg scan_seg(const ScanArgs& a, int bh, int seg) {
  const size_t per_c = (size_t)a.DHQK * a.DHHV, count = (size_t)a.n_bh * (a.nseg - 1), idx = (size_t)bh * (a.nseg - 1) + seg;
  return {a.seg + idx * per_c, a.seg + count * per_c + idx * a.DHQK};
}

// The consumer role of the scan kernel (see there).  NDB = 0 or 1: this wave also carries the normaliser vector of the
// first or second 32 of its 64 state rows, NDB = -1: it does not (copies of the role rather than a branch around matrix
// instructions, which would make the compiler keep those accumulators in scratch memory).
// `run`: runs this workgroup has made, `chunk`: chunks it has finished; they select the LDS buffer and the slots of the tables.
template <int RT, int WT, bool F16, bool REP, bool SEG, int NDB>
__device__ __forceinline__ void scan_consumer(const ScanArgs& a, const uint16_t* bufs, const float* gl, const uint16_t* nB,
                                              int wave, int lane, const ScanJob& job, int& run, int& chunk) {
  constexpr int WC = WT / 32;
  constexpr int NWC = (RT / 64) * WC;
  constexpr int XELEMS = kChunk * RT, YELEMS = kChunk * WT;
  constexpr int BUF = XELEMS + YELEMS;
  const int DHQK = a.DHQK, DHHV = a.DHHV, NC = a.NC;
  ScanRuns<REP> runs;
  runs.set(job.it_lo, job.it_hi, job.it_rep);
  const int bh = job.bh, seg = job.seg, total = runs.total;
  const int tile = job.bx + (DHQK / RT) * job.by, d_tile = job.bx * RT, w_tile = job.by * WT;
  const bool is_end = job.end & 1;
  constexpr bool WITH_N = NDB >= 0;  // (forward only)
  const bool backward = !WITH_N && a.backward;
  const int c_base = backward ? NC - 1 : 0, c_step = backward ? -1 : 1;
  // slot and position of the running chunk among the kept states, carried along: divisions by the stride in the loop
  // take as long as half its matrix instructions
  int st_slot = (c_base + runs.it_lo * c_step) / a.stride, st_pos = (c_base + runs.it_lo * c_step) % a.stride;
  constexpr int DB = WITH_N ? NDB : 0;
  const int wr = wave / WC, wc = wave % WC;
  const int r = lane & 31, h = lane >> 5;
  const int d_wave = d_tile + wr * 64, w_wave = w_tile + wc * 32;
  f32x16 acc[2], accn;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = accn[i] = 0.f;
  if (a.init != nullptr && (!SEG || a.seg_phase != 1)) {
    const float* const src = a.init + ((size_t)bh * DHQK + d_wave + 4 * h) * DHHV + w_wave + r;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] = src[(size_t)(32 * db + 8 * (i / 4) + (i % 4)) * DHHV];
  }
  // normaliser vector: the waves of the first 32 value columns of the first column tile carry it as three partial
  // columns (lanes r = 0, 1, 2) of one more accumulator pair, see write_tables
  if (WITH_N && a.n_init != nullptr && (!SEG || a.seg_phase != 1) && r == 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) accn[i] = a.n_init[(size_t)bh * DHQK + d_wave + 32 * DB + 8 * (i / 4) + 4 * h + (i % 4)];
  }
  const size_t seg_ofs = ((size_t)tile * NWC + wave) * 2048 + lane * 4;
  if (SEG && a.seg_phase == 2) {
    // the state before this segment: the segments in front of it, each decayed over what lies between
    for (int x = 0; x < seg; ++x) {
      float dec = 1.f;
      for (int k = lane; k < a.seg_len; k += kWave) {
        const int itx = x * a.seg_len + k;
        dec *= a.gbar[(size_t)bh * NC + (a.backward ? NC - 1 - itx : itx)];
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) dec *= __shfl_xor(dec, o);
      const ScanSeg ss = scan_seg(a, bh, x);
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const f32x4 v = *(const f32x4*)(ss.c + seg_ofs + (db * 4 + g4) * 256);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[db][4 * g4 + e] = acc[db][4 * g4 + e] * dec + v[e];
        }
      if (WITH_N) {
        // (four values a load, of all lanes: one at a time under r == 0 they were sixteen trips to memory in a row)
        const float* const nsrc = ss.n + d_wave + 32 * DB + 4 * h;
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const f32x4 v = *(const f32x4*)(nsrc + 8 * g4);
#pragma unroll
          for (int e = 0; e < 4; ++e) accn[4 * g4 + e] = accn[4 * g4 + e] * dec + (r == 0 ? v[e] : 0.f);
        }
      }
    }
  }
  const ScanTrOff offA0 = scan_tr_offsets<RT>(wr * 64, lane);
  const ScanTrOff offA1 = scan_tr_offsets<RT>(wr * 64 + 32, lane);
  const ScanTrOff offB = scan_tr_offsets<WT>(wc * 32, lane);
  // ---- the state before chunk `it` as operand fragments, at the kept boundaries only: forward the state before every
  // stride-th chunk, backward the gradient of the state after the last chunk of every group of `stride` chunks (and after
  // the last chunk of the sequence); slot c / stride either way.  A state known to be zero is not written if nobody reads it.
  auto emit_state = [&](int it) __attribute__((always_inline)) {
    const int c = c_base + it * c_step;
    const bool keep = (!SEG || a.seg_phase != 1) && (backward ? (c == NC - 1 || st_pos == a.stride - 1) : st_pos == 0) &&
                      !(it == 0 && a.skip_zero && a.init == nullptr);
    if (keep) {
      const size_t ND = DHQK / 16, NWB = DHHV / 32;
      const size_t NCS = (size_t)(NC + a.stride - 1) / a.stride;
      u32x4* st = (u32x4*)a.states + ((size_t)bh * NCS + st_slot) * NWB * ND * 64;
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        const size_t W32 = w_wave / 32, D16 = (d_wave + 32 * db) / 16;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          u32x4 f;
#pragma unroll
          for (int e = 0; e < 4; ++e) f[e] = pack2<F16>(acc[db][8 * half + 2 * e], acc[db][8 * half + 2 * e + 1]);
          // non-temporal: the fragments are read by a later kernel; kept out of the L2 they do not evict the K/V
          // rows the tiles of a head share
          __builtin_nontemporal_store(f, st + (W32 * ND + D16 + half) * 64 + lane);
        }
      }
    }
  };
  // ---- n before chunk `it`, as its three partial vectors [3][DHQK] (the consumer of the states adds them up)
  auto emit_n = [&](int it) __attribute__((always_inline)) {
    if (r < 3 && (!SEG || a.seg_phase != 1)) {
      float* dst = a.nstates + (((size_t)bh * NC + it) * 3 + r) * DHQK + d_wave + 32 * DB + 4 * h;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *(float4*)(dst + 8 * g4) = make_float4(accn[4 * g4], accn[4 * g4 + 1], accn[4 * g4 + 2], accn[4 * g4 + 3]);
    }
  };
  for (int p = 0; p < total; ++p) {
    const int it = runs.it(p);
    const bool rest = runs.rest(p);
    __syncthreads();  // run p staged by the producers
    if (!rest) {
      emit_state(it);
      st_pos += c_step;
      if (st_pos == a.stride) {
        st_pos = 0;
        ++st_slot;
      } else if (st_pos < 0) {
        st_pos = a.stride - 1;
        --st_slot;
      }
      const float g = gl[chunk & 3];
      acc[0] *= g;
      acc[1] *= g;
      if (WITH_N) {
        emit_n(it);
        accn *= g;
      }
    }
    // ---- accumulate X^T (scale . Y) over the positions of the chunk
    const uint16_t* Xs = bufs + (run & 1) * BUF;
    const uint16_t* Yh = Xs + XELEMS;
    const uint16_t* nBp = nB + (chunk % 3) * (kChunk * 3) + h * 24 + min(r, 2) * 8;
#pragma unroll
    for (int js = 0; js < kChunk / 16; ++js) {
      const Frag A0 = scan_tr_frag<RT>(Xs, 16 * js, offA0), A1 = scan_tr_frag<RT>(Xs, 16 * js, offA1);
      const Frag Bh = scan_tr_frag<WT>(Yh, 16 * js, offB);
      mfma32<F16>(acc[0], A0, Bh);
      mfma32<F16>(acc[1], A1, Bh);
      if (WITH_N) {
        Frag Bn;
        Bn.u = *(const uint4*)(nBp + js * 48);
        // (a second run adds nothing: the three parts carry the whole scale)
        if (r >= 3 || rest) Bn.u = make_uint4(0, 0, 0, 0);
        mfma32<F16>(accn, DB == 0 ? A0 : A1, Bn);
      }
    }
    ++run;
    if (runs.last(p)) ++chunk;
  }
  if (job.end >> 1) {
    emit_state((job.end >> 1) - 1);
    if (WITH_N) emit_n((job.end >> 1) - 1);
  }
  if (SEG && a.seg_phase == 1) {
    const ScanSeg ss = scan_seg(a, bh, seg);
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const f32x4 v = {acc[db][4 * g4], acc[db][4 * g4 + 1], acc[db][4 * g4 + 2], acc[db][4 * g4 + 3]};
        *(f32x4*)(ss.c + seg_ofs + (db * 4 + g4) * 256) = v;
      }
  } else if (a.final_out != nullptr && is_end) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = d_wave + 32 * db + 8 * (i / 4) + 4 * h + (i % 4);
        a.final_out[((size_t)bh * DHQK + d) * DHHV + w_wave + r] = acc[db][i];
      }
  }
  if (WITH_N && (SEG && a.seg_phase == 1 || (a.n_final != nullptr && is_end))) {
    float* const dst = SEG && a.seg_phase == 1 ? scan_seg(a, bh, seg).n : a.n_final + (size_t)bh * DHQK;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      // the three partial columns live in lanes r = 0, 1, 2 of either half wave
      const float x = accn[i];
      const float sum = __shfl(x, 32 * h) + __shfl(x, 32 * h + 1) + __shfl(x, 32 * h + 2);
      if (r == 0) dst[d_wave + 32 * DB + 8 * (i / 4) + 4 * h + (i % 4)] = sum;
    }
  }
}

// RT x WT state tile, one chunk of 128 positions per run.  REP: the late chunks run twice; SEG: the sequence is cut into
// segments (both compile-time: tested per run they cost the plain scan 6 %, 331 against 311 us at B = 4, S = 16384).
//
// The workgroup has two kinds of waves, NWC of each: CONSUMER waves own a 64 x 32 block of the state tile in their
// accumulators and do nothing but fragment reads, matrix instructions, the decay and the emission of the state;
// PRODUCER waves fetch the rows, scale and round them and write them into the LDS buffer the consumers will read
// next, keep the normaliser operand and the scale table.  The two instruction streams of a SIMD that limit each other
// when every wave does everything (conversion arithmetic against matrix instructions) then belong to different waves
// and overlap; four waves per SIMD instead of two.
//
// The workgroups are persistent (MANY; a launch of no more jobs than fit the chip keeps the plain form, whose loop has no
// cursors).  As many run as fit by LDS, one per CU (tiles of 64 x 64: two); with more than kScanRounds jobs for each the grid
// has more workgroups than are resident, each of which ends after its share.  Where one fills a CU, a tile of eight chunks spent
// a third of its time on filling the pipeline and on its last stores with the CU otherwise idle.  Now the next tile's rows are on their way meanwhile.  Without a last state the
// chunks behind the last kept boundary (in front of the first one) are not run: only n, for its own tiles, is wanted there.
// Both together, us for a forward and backward call: 128 heads of 1024, 256/512, with layer norm 729 -> 665, 64 heads of 1000
// 330 -> 302, 128 heads of 2048, 128/256 500 -> 487; 128 heads of 2048 with the last state, forward 418 -> 416.
template <int RT, int WT, bool F16, bool REP, bool SEG, bool MANY>
__global__ __launch_bounds__(128 * (RT / 64) * (WT / 32)) void scan_roles_kernel(ScanArgs a, int n_rounds) {
  if constexpr (!REP) {
    if (a.unless != nullptr && __builtin_amdgcn_readfirstlane(*a.unless) != 0) return;
  }
  constexpr int WC = WT / 32;
  constexpr int NWC = (RT / 64) * WC;     // consumer waves (and as many producer waves)
  constexpr int NTP = 64 * NWC;           // producer threads
  constexpr int XU = RT / 8, YU = WT / 8; // 16-byte units per row
  constexpr int XV = kChunk * XU / NTP;   // 16-byte vectors per producer thread per chunk
  constexpr int YV = kChunk * YU / NTP;
  constexpr int XRG = NTP / XU;           // rows one sweep of the producers covers (X); a thread's rows are XRG apart
  constexpr int YRG = NTP / YU;
  constexpr int XELEMS = kChunk * RT, YELEMS = kChunk * WT;
  constexpr int BUF = XELEMS + YELEMS;    // elements per LDS buffer
  static_assert(XV >= 1 && YV >= 1 && XRG % 4 == 0 && YRG % 4 == 0, "tile shape does not fit the staging pattern");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  uint16_t* bufs = (uint16_t*)smem_raw;                 // [2][X | Y]
  float* gl = (float*)(bufs + 2 * BUF);                 // [4] decay factors, by chunk of this workgroup
  float* scl = gl + 4;                                  // [2][128] row scales, likewise
  uint16_t* nB = (uint16_t*)(scl + 2 * kChunk);         // [3][128 / 8][3][8] the row scales as a matrix operand (below)
  ScanJob* jobs = (ScanJob*)(nB + 3 * kChunk * 3);      // [kScanRounds]

  // the wave index is made scalar so that branches on it are scalar branches
  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const bool producer = wave_all < NWC;
  const int wave = producer ? wave_all : wave_all - NWC;
  const int tid = wave * 64 + lane;                     // index inside the own group of waves
  const int G = gridDim.x;
  int vid = blockIdx.x;
  if (G % 8 == 0) vid = (vid % 8) * (G / 8) + vid / 8;  // consecutive ids share an XCD (and its L2)
  ScanJob job0 = {0, 0, 0, 0, 0, 0, 0, 0};  // !MANY: the only one
  if constexpr (MANY) {
    for (int rd = wave_all; rd < n_rounds; rd += 2 * NWC) {
      const ScanJob job = scan_decode<RT, WT, REP, SEG>(a, rd, vid, lane);
      if (lane == 0) jobs[rd] = job;
    }
    __syncthreads();
  } else {
    job0 = scan_decode<RT, WT, REP, SEG>(a, 0, vid, lane);
  }

  if (producer) {
    // ======================================================================================= producer waves
    const int DHQK = a.DHQK, DHHV = a.DHHV, S = a.S, NC = a.NC;
    const size_t Sp = (size_t)NC * kChunk;
    const int c_base = a.backward ? NC - 1 : 0, c_step = a.backward ? -1 : 1;
    const int xrow = tid / XU, yrow = tid / YU;  // first row of this thread inside a chunk; further rows XRG / YRG apart
    const int xcol = (tid % XU) * 8, ycol = (tid % YU) * 8;
    // byte offsets of the first row inside a chunk of the operands
    const uint32_t xofs = (uint32_t)(xrow * DHQK + xcol) * 2, yofs = (uint32_t)(yrow * DHHV + ycol) * 2;
    // LDS store offsets of the first row (elements); the rows of a thread are a multiple of 4 apart: same swizzle
    const int xst = xrow * RT + (((tid % XU) ^ scan_swz<XU>(xrow)) << 3);
    const int yst = yrow * WT + (((tid % YU) ^ scan_swz<YU>(yrow)) << 3);

    // (Scalar bases and 32-bit offsets inside a chunk: with a 64-bit product for every row, and with the bases worked out from the
    // job's indexes in every run, the producers' instructions were what a narrow tile took.  256/320, 16 heads of 512 / of 2048 with
    // the last state: 14.2 -> 13.1, 30.4 -> 28.1 us; 40 heads of 256/512, 512 positions, backward 23.3 -> 22.3.)
    // The runs of all jobs of this workgroup form one sequence, and the producers work ahead of it without regard to where a
    // job ends: run P + 3 is requested and run P + 1 staged while run P is multiplied, the scales of the chunk three ahead
    // are requested.  Two cursors walk the jobs, one over runs and one over chunks; past the last job they stay where they
    // are (the requests are unconditional: a conditional one makes the compiler keep the registers in scratch memory).
    int r_rd = -1, r_p = -1, r_bh = job0.bh, r_bx = job0.bx, r_by = job0.by, r_par = 0;  // run cursor
    const uint16_t* r_x = a.X + (size_t)r_bh * S * DHQK + r_bx * RT;
    const uint16_t* r_y = a.Y + (size_t)r_bh * S * DHHV + r_by * WT;
    ScanRuns<REP> rr;
    rr.set(job0.it_lo, job0.it_hi, job0.it_rep);
    int k_rd = -1, k_bh = job0.bh, k_by = job0.by, k_it = job0.it_lo - 1, k_hi = job0.it_hi;  // chunk cursor
    // a run's properties travel with it: bit 0 there is one, 1 second run of its chunk, 2 last run of its chunk, 3 its slot in
    // the scale table
    auto next_run = [&]() -> int {
      if (r_p + 1 < rr.total) {
        ++r_p;
      } else {
        if constexpr (!MANY) return 0;
        int lo, hi, rep;
        do {
          if (r_rd + 1 >= n_rounds) return 0;
          ++r_rd;
          lo = __builtin_amdgcn_readfirstlane(jobs[r_rd].it_lo);
          hi = __builtin_amdgcn_readfirstlane(jobs[r_rd].it_hi);
          rep = __builtin_amdgcn_readfirstlane(jobs[r_rd].it_rep);
        } while (lo == hi);
        r_bh = __builtin_amdgcn_readfirstlane(jobs[r_rd].bh);
        r_bx = __builtin_amdgcn_readfirstlane(jobs[r_rd].bx);
        r_by = __builtin_amdgcn_readfirstlane(jobs[r_rd].by);
        rr.set(lo, hi, rep);
        r_p = 0;
        r_x = a.X + (size_t)r_bh * S * DHQK + r_bx * RT;
        r_y = a.Y + (size_t)r_bh * S * DHHV + r_by * WT;
      }
      const bool last = rr.last(r_p);
      const int m = 1 | (rr.rest(r_p) ? 2 : 0) | (last ? 4 : 0) | (r_par << 3);
      if (last) r_par ^= 1;
      return m;
    };
    auto next_chunk = [&]() -> bool {
      if (k_it + 1 < k_hi) {
        ++k_it;
        return true;
      }
      if constexpr (!MANY) return false;
      int lo, hi;
      do {
        if (k_rd + 1 >= n_rounds) return false;
        ++k_rd;
        lo = __builtin_amdgcn_readfirstlane(jobs[k_rd].it_lo);
        hi = __builtin_amdgcn_readfirstlane(jobs[k_rd].it_hi);
      } while (lo == hi);
      k_bh = __builtin_amdgcn_readfirstlane(jobs[k_rd].bh);
      k_by = __builtin_amdgcn_readfirstlane(jobs[k_rd].by);
      k_it = lo;
      k_hi = hi;
      return true;
    };

    // ---- row scales (forward: abar_j; backward: bbar_t / sqrt(DHQK) / (nrow_t + eps)) go through a table in LDS:
    // every thread fetches the factor of ONE row of a chunk three chunks before that chunk is staged (first in its
    // batch of loads, so that waiting for it does not wait for the rows requested with it) and writes the table entry
    // one chunk later; positions past the end of the sequence get 0 and so neither feed the state nor the normaliser.
    // The decay factor of the chunk rides along.
    const int srow = tid & (kChunk - 1);
    const float* const nrow_or_dummy = a.nrow != nullptr ? a.nrow : a.scale_a;
    float s_raw = 0.f, s_nrm = 1.f, s_g = 0.f;
    int s_lim = 0;       // rows of the chunk that lie inside the sequence
    bool s_n = false;    // whether the chunk's tile carries n
    auto load_scales = [&](bool there) {  // of the chunk cursor's chunk
      const int c = __builtin_amdgcn_readfirstlane(c_base + max(k_it, 0) * c_step);
      const size_t o = (size_t)k_bh * NC + c;
      s_raw = (a.scale_a + o * kChunk)[(uint32_t)srow];
      s_nrm = (nrow_or_dummy + o * kChunk)[(uint32_t)srow];
      s_g = (a.gbar + o)[(uint32_t)opaque(0)];
      s_lim = there ? S - c * kChunk : 0;
      s_n = there && a.nstates != nullptr && k_by == 0;
    };
    auto scale_value = [&]() {  // the table entry of row srow from the fetched values
      float sn = srow < s_lim ? s_raw : 0.f;
      if (a.backward) {
        sn *= a.qk_scale;
        if (a.nrow != nullptr) sn /= (s_nrm + a.eps);
      }
      return sn;
    };

    // The normaliser recurrence n_c = gbar_c n_{c-1} + sum_j abar_j k_j rides on the matrix pipe of the consumers: the
    // row scale of every position, split exactly into three 16-bit parts, forms three columns of a B operand
    // (position 8b + e of a chunk, part r, at [b][r][e]); K^T times it gives sum_j abar_j k_j in three partial columns
    // whose sum carries 24 bits of every abar_j.  Written two chunks before the chunk is multiplied, three slots.
    auto write_tables = [&](int chunk) {
      // (two waves have all rows: the others leave the division of the backward out)
      if (NTP == kChunk || wave < kChunk / 64) {
        const float sn = scale_value();
        scl[(chunk & 1) * kChunk + srow] = sn;
        if (tid == 0) gl[chunk & 3] = s_g;
        if (s_n) {
          uint16_t* dst = nB + (chunk % 3) * (kChunk * 3) + (srow >> 3) * 24 + (srow & 7);
          const uint16_t p0 = f32_to_elem<F16>(sn);
          const float r1 = sn - elem_to_f32<F16>(p0);
          const uint16_t p1 = f32_to_elem<F16>(r1);
          const uint16_t p2 = f32_to_elem<F16>(r1 - elem_to_f32<F16>(p1));
          dst[0] = p0;
          dst[8] = p1;
          dst[16] = p2;
        }
      }
    };

    // two register sets, by run parity (macros, not lambdas: with the arrays captured by reference the compiler keeps
    // them in scratch memory)
    u32x4 xr0[XV], yr0[YV], xr1[XV], yr1[YV];
    // The prefetch only LOADS: any arithmetic on a loaded value here would make the wave wait for the whole batch.
#define MLSTM_SCAN_PREFETCH(SET)                                                                                 \
  {                                                                                                              \
    const int t0_ = __builtin_amdgcn_readfirstlane((c_base + rr.it(max(r_p, 0)) * c_step) * kChunk);             \
    const int last_ = min(kChunk - 1, S - 1 - t0_); /* rows past the end re-read the last row; their scale is 0 */ \
    const char* const xb_ = (const char*)(r_x + (size_t)t0_ * DHQK);                                             \
    const char* const yb_ = (const char*)(r_y + (size_t)t0_ * DHHV);                                             \
    const uint32_t xl_ = (uint32_t)(last_ * DHQK + xcol) * 2, yl_ = (uint32_t)(last_ * DHHV + ycol) * 2;         \
    _Pragma("unroll") for (int v = 0; v < XV; ++v)                                                               \
      xr##SET[v] = *(const u32x4*)(xb_ + min(xofs + (uint32_t)(v * XRG * 2) * (uint32_t)DHQK, xl_));              \
    _Pragma("unroll") for (int v = 0; v < YV; ++v)                                                               \
      yr##SET[v] = *(const u32x4*)(yb_ + min(yofs + (uint32_t)(v * YRG * 2) * (uint32_t)DHHV, yl_));              \
  }
    // registers -> LDS buffer SET (Y rows scaled in fp32, then rounded; second runs: the remainder of that rounding)
#define MLSTM_SCAN_STAGE(SET, meta_)                                                                             \
  {                                                                                                              \
    uint16_t* Xs = bufs + (SET) * BUF;                                                                           \
    uint16_t* Yh = Xs + XELEMS;                                                                                  \
    const float* scur = scl + (((meta_) >> 3) & 1) * kChunk;                                                     \
    const bool rest_ = REP && ((meta_) & 2);                                                                     \
    _Pragma("unroll") for (int v = 0; v < XV; ++v) *(u32x4*)(Xs + xst + v * XRG * RT) = xr##SET[v];              \
    _Pragma("unroll") for (int v = 0; v < YV; ++v) {                                                             \
      const uint32_t in[4] = {yr##SET[v][0], yr##SET[v][1], yr##SET[v][2], yr##SET[v][3]};                       \
      uint32_t hi[4];                                                                                            \
      const float sc = scur[yrow + v * YRG];                                                                     \
      _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                                            \
        float e0 = lo2<F16>(in[e]) * sc;                                                                         \
        float e1 = hi2<F16>(in[e]) * sc;                                                                         \
        /* both runs round the same fp32 products: the product and its conversion to float16 may be fused in */  \
        /* one of them, and the remainder would then belong to another head */                                   \
        if constexpr (F16) asm("" : "+v"(e0), "+v"(e1));                                                         \
        hi[e] = pack2<F16>(e0, e1);                                                                              \
        if (rest_) hi[e] = pack2<F16>(e0 - lo2<F16>(hi[e]), e1 - hi2<F16>(hi[e]));                               \
      }                                                                                                          \
      *(uint4*)(Yh + yst + v * YRG * WT) = make_uint4(hi[0], hi[1], hi[2], hi[3]);                               \
    }                                                                                                            \
  }

    // ---- prologue: tables of the first two chunks, runs 0 and 1 in registers, run 0 staged, run 2 requested
    int chunk = 0;
    load_scales(next_chunk());
    write_tables(0);
    load_scales(next_chunk());
    write_tables(1);
    load_scales(next_chunk());  // written at the last run of the first chunk
    bool more = next_chunk();
    int m0 = next_run();
    MLSTM_SCAN_PREFETCH(0)
    int m1 = next_run();
    MLSTM_SCAN_PREFETCH(1)
    __syncthreads();  // tables visible
    MLSTM_SCAN_STAGE(0, m0)
    int m2 = next_run();
    MLSTM_SCAN_PREFETCH(0)
    int m3 = next_run();

    // one run, of properties m0; the next one and the one two after that use LDS buffer and register set OTHER
#define MLSTM_SCAN_BODY(OTHER)                                                                                   \
  {                                                                                                              \
    /* this run is staged; the consumers are done with the one before it, whose buffer is staged into next */    \
    __syncthreads();                                                                                             \
    if (m0 & 4) {                                                                                                \
      /* Table entry of the chunk after the next (its factors were fetched one chunk ago) into the slot of the */ \
      /* present one, all of whose runs have been staged; it is read from the next run on.  Then the factors */  \
      /* of the chunk after that are requested, first in this run's batch of loads. */                           \
      write_tables(chunk + 2);                                                                                   \
      load_scales(more);                                                                                         \
    }                                                                                                            \
    if (m1 & 1) MLSTM_SCAN_STAGE(OTHER, m1)                                                                      \
    MLSTM_SCAN_PREFETCH(OTHER)                                                                                   \
    /* the cursors move on when everything is on its way */                                                      \
    if (m0 & 4) {                                                                                                \
      more = next_chunk();                                                                                       \
      ++chunk;                                                                                                   \
    }                                                                                                            \
    m0 = m1;                                                                                                     \
    m1 = m2;                                                                                                     \
    m2 = m3;                                                                                                     \
    m3 = next_run();                                                                                             \
  }
    while (m0 & 1) {
      MLSTM_SCAN_BODY(1)
      if (m0 & 1) MLSTM_SCAN_BODY(0)
    }
#undef MLSTM_SCAN_BODY
#undef MLSTM_SCAN_STAGE
#undef MLSTM_SCAN_PREFETCH
  } else {
    // ======================================================================================= consumer waves
    int run = 0, chunk = 0;
    __syncthreads();  // the producers' prologue barrier
    for (int rd = 0; rd < (MANY ? n_rounds : 1); ++rd) {
      ScanJob job = job0;
      if constexpr (MANY) {
        int* const w = (int*)&job;
#pragma unroll
        for (int x = 0; x < (int)(sizeof(ScanJob) / sizeof(int)); ++x) w[x] = __builtin_amdgcn_readfirstlane(((const int*)(jobs + rd))[x]);
      }
      if (job.it_lo == job.it_hi && job.end == 0) continue;
      // the normaliser vector rides with two waves of every 64 state rows in the first column tile: one for the first and one for
      // the second 32 rows, a SIMD each (with both row groups on the same two SIMDs 128 chunks of the forward took 1.5 % longer)
      const bool with_n = (a.nstates != nullptr) && job.by == 0;
      const int nd = wave % WC - (NWC == 8 ? 2 * (wave / WC) : 0);
      if (with_n && nd == 0)
        scan_consumer<RT, WT, F16, REP, SEG, 0>(a, bufs, gl, nB, wave, opaque(lane), job, run, chunk);
      else if (with_n && nd == 1)
        scan_consumer<RT, WT, F16, REP, SEG, 1>(a, bufs, gl, nB, wave, opaque(lane), job, run, chunk);
      else
        scan_consumer<RT, WT, F16, REP, SEG, -1>(a, bufs, gl, nB, wave, opaque(lane), job, run, chunk);
    }
  }
}

static size_t scan_roles_smem(int RT, int WT) {
  return (size_t)2 * kChunk * (RT + WT) * 2 + (size_t)(4 + 2 * kChunk) * 4 + (size_t)3 * kChunk * 3 * 2 + kScanRounds * sizeof(ScanJob);
}
template <int RT, int WT, bool F16, bool REP, bool SEG, bool MANY>
static const char* launch_scan_roles_m(const ScanArgs& a, int G, int n_rounds, hipStream_t stream) {
  constexpr int NW = (RT / 64) * (WT / 32);
  static LdsLimit lds;
  if (!lds.allow((const void*)scan_roles_kernel<RT, WT, F16, REP, SEG, MANY>, scan_roles_smem(RT, WT)))
    return "scan: cannot raise the dynamic LDS limit";
  hipLaunchKernelGGL((scan_roles_kernel<RT, WT, F16, REP, SEG, MANY>), dim3(G), dim3(128 * NW), scan_roles_smem(RT, WT), stream, a, n_rounds);
  return nullptr;
}
template <int RT, int WT, bool F16, bool REP, bool SEG>
static const char* launch_scan_roles_f(ScanArgs a, int BH, hipStream_t stream) {
  const long long n_jobs = (long long)(a.DHQK / RT) * (a.DHHV / WT) * BH * (a.seg_phase == 1 ? a.nseg - 1 : a.nseg);
  if (n_jobs >= (1ll << 30)) return "scan: too many state tiles";
  const int cus = device_cu_count();
  if (cus <= 0) return "scan: cannot read the number of compute units";
  a.n_jobs = (int)n_jobs;
  const int fit = cus * (int)(160 * 1024 / scan_roles_smem(RT, WT));
  // Few tiles more than fit: where a tile is smaller than 128 x 128 a workgroup for each, which start as others end, is the faster
  // form (fixed shares make the last of them late); not with one tile a head.  Us, persistent / a workgroup each, with the last
  // state, without, backward: 256/320, 32 heads (1.25 tiles for each that fits) of 512 24.2 14.3 16.8 / 22.0 12.0 17.1, of 2048
  // 52.4 41.6 41.4 / 50.0 37.1 41.2; 64/384, 112 heads (1.3) of 2048 70.8 58.7 66.6 / 66.5 56.6 67.8; 192/192, 64 heads (1.1) of 2048
  // 68.6 53.8 51.6 / 63.9 49.5 49.7; but 128/192, 168 heads (2.0) of 2048 71.1 60.2 62.1 / 72.5 62.7 65.0 and 64/64, 640 heads (1.25)
  // of 2048 96.1 84.5 83.1 / 104.6 89.7 88.1.
  const bool few = (RT < 128 || WT < 128) && a.n_jobs > BH && 5ll * a.n_jobs < 7ll * fit;
  if (a.n_jobs <= fit || (!SEG && few)) return launch_scan_roles_m<RT, WT, F16, REP, SEG, false>(a, a.n_jobs, 1, stream);
  if constexpr (SEG) {
    return "scan: more segments than the chip holds";
  } else {
    const int least = (a.n_jobs + kScanRounds - 1) / kScanRounds;
    int G = fit > least + 7 ? fit : least + 7;
    if (G >= 8) G -= G % 8;
    return launch_scan_roles_m<RT, WT, F16, REP, SEG, true>(a, G, (a.n_jobs + G - 1) / G, stream);
  }
}
template <int RT, int WT, bool F16>
static const char* launch_scan_roles_s(const ScanArgs& a, int BH, hipStream_t stream) {
  if (a.nseg > 1)
    return a.part == 1 ? launch_scan_roles_f<RT, WT, F16, true, true>(a, BH, stream) : launch_scan_roles_f<RT, WT, F16, false, true>(a, BH, stream);
  return a.part == 1 ? launch_scan_roles_f<RT, WT, F16, true, false>(a, BH, stream) : launch_scan_roles_f<RT, WT, F16, false, false>(a, BH, stream);
}
template <int RT, int WT>
static const char* launch_scan_roles_t(const ScanArgs& a, int BH, hipStream_t stream) {
  return a.f16 ? launch_scan_roles_s<RT, WT, true>(a, BH, stream) : launch_scan_roles_s<RT, WT, false>(a, BH, stream);
}

const char* launch_scan(const ScanArgs& a_in, int BH, bool hilo, hipStream_t stream) {
  ScanArgs a = a_in;
  a.part = 0;
  a.n_bh = BH;
  a.nseg = 1;
  a.seg_len = a.NC;
  a.seg_phase = 0;
  // Chunks that are run at all: without a last state those up to the last kept boundary (forward), down to the first one
  // (backward), and for n, which is kept at every chunk, up to the last chunk.
  a.end_c = a.end_n = a.NC;
  if (a.final_out == nullptr && a.stride >= 1) {
    a.end_c = a.backward ? (a.NC > a.stride ? a.NC - a.stride : 0) : (a.NC - 1) / a.stride * a.stride;
    if (a.n_final == nullptr) a.end_n = a.NC - 1;
  }
  if (a.DHQK % 64 != 0 || a.DHHV % 64 != 0) return "scan: DHQK and DHHV must be multiples of 64";
  if (a.stride < 1 || a.stride > kMaxStateStride) return "scan: state stride out of range";
  // (up to one group of chunks and no state from outside: nothing to run and nothing to write)
  if (a.skip_zero && a.init == nullptr && a.final_out == nullptr && a.nstates == nullptr && a.end_c == 0) return nullptr;
  const bool r128 = a.DHQK % 128 == 0;
  bool w128 = a.DHHV % 128 == 0;
  // Segments (see the top of the file): the number of them, of those that fit the chip beside each other, that the two launches
  // take the least time with.  Their states go through the caller's scratch (an output that is written later), which has to
  // hold them.  Fixed time, time for a chunk of a segment and for a segment in front, from sweeps of 1 to 16 segments, and 10 %
  // for what they leave out.  us, one scan in one piece / in the segments that this takes: 4 heads of 64/64, 2000 positions 37.0 / 30.5,
  // 4000 62.3 / 34.5, 10000 135.6 / 42; 32 heads of 64/128, 4000 62.4 / 43.3; 16 heads of 128/256, 4000 50.0 / 47.1; 8 heads of 256/512,
  // 10000 130.9 / 102.4, but 4000 50.1 / 53.4 (tiles of half the width in one piece).  With a backward the launches of a short call are what
  // its host takes the longest for (4 heads of 64/64, 2048 positions, forward and backward 102 / 107): 8 us have to be gained there.
  {
    const int tiles = (a.DHQK / (r128 ? 128 : 64)) * (a.DHHV / (w128 ? 128 : 64));
    const bool wide = r128 && w128;
    const int fit = device_cu_count() / (BH * tiles);
    const bool halves = wide && 2ll * BH * tiles <= device_cu_count();  // (see below)
    const float one_piece = wide ? (halves ? 4.f + 1.6f * a.NC : 12.f + 1.9f * a.NC) : 12.f + (r128 ? 1.4f : 1.57f) * a.NC;
    float best = a.with_backward ? fminf(0.9f * one_piece, one_piece - 8.f) : 0.9f * one_piece;
    int len = 0;
    for (int n = 2; n <= (wide ? 8 : 16) && n <= fit && a.by_batch; ++n) {
      const int l = (a.NC + n - 1) / n;
      const float t = wide ? 16.f + 4.f * l + 1.2f * n : 20.f + 2.8f * l + 0.55f * n;
      if (t < best && (size_t)BH * (n - 1) * ((size_t)a.DHQK * a.DHHV + a.DHQK) * sizeof(float) <= a.seg_bytes) {
        best = t;
        len = l;
      }
    }
    if (len > 0 && a.seg != nullptr) {
      a.seg_len = len;
      a.nseg = (a.NC + len - 1) / len;
    }
    // Late chunks in a second run whatever their number: sequences of four chunks; where the kernels may be chosen by the heads
    // of the call, all in segments, whose other kernel would walk the late chunks of all segments in one piece; a scan in one piece up
    // to 24 chunks, or of any number while the tiles do not fill the chip; with the sigmoid gate, where all chunks are late, while they do not
    // and the rows that run twice are few.
    // us for a forward with the last state, a launch more / so, the last chunk late / all of them: in one piece, 256/512, 8 heads of 700
    // 49.3 52.2 / 39.5 44.4, of 2000 56.4 82.6 / 54.0 70.2, 64 of 1000 117.5 149.9 / 112.4 132.3, 96 of 3000 448 558 / 446 547, but 96 of 8000 all
    // late 1386 / 1414; 64/64, 4 heads of 1000 37.2 50.3 / 35.7 45.4.  In segments, 256/512, 8 heads of 10000 201 370 / 199 257; 16 of
    // 128/256, 4000 81.0 149 / 78.7 86.7; 64/64, 4 heads of 10000 63.3 282 / 60.1 71.3, 12 of 4000 56.9 141 / 54.2 57.1, 32 of 2000 49.3 87.6 / 46.4
    // 48.7; 64/128, 64 of 4000 124 183 / 121 144; 128/64, 32 of 3000 74.5 121 / 72.3 75.3 (these three in one piece and a launch more 81 to 186 with
    // all late).  Sigmoid gate in one piece: 128/128, 40 heads of 2000 87.0 / 83.3, 256/512, 8 of 2600 98.7 / 91.5, 256/256, 24 of 2600 136.7 /
    // 134.8, but 256/512, 24 of 1100 68.9 / 70.7, 256/256, 40 of 1100 66.8 / 68.6, 128/256, 64 of 2000 105.1 / 109.4, 256/512, 64 of 4000 473 / 487.
    const bool fills = (long long)BH * tiles >= device_cu_count();
    const bool rows = wide && (long long)BH * (a.DHQK + a.DHHV) >= 48ll * device_cu_count();
    const bool one_launch = len > 0 ? a.seg != nullptr : a.all_remainder ? !fills && !rows : !fills || a.NC <= 24;
    a.repeat_all = a.NC <= 4 || (a.by_batch && one_launch);
  }
  // Tiles of half the width where those of both halves still have a CU each: the walk over the chunks is what the launch
  // takes then, and half the columns make a chunk a quarter shorter (256/512, us, 128 / 64 columns: 8 heads of 317 positions
  // with the last state 20.5 / 16.1, of 2048 without 33.6 / 26.2; 16 heads of 10000 157 / 118).  With more tiles than CUs
  // the rows are read twice for nothing (32 heads of 2048: 37.6 / 44.9); half the rows instead gain less (17.5, 26.3, 128).
  const int ncol = a.DHHV / 128 * (a.DHQK / (r128 ? 128 : 64));
  if (w128 && a.nseg == 1 && 2ll * BH * ncol <= device_cu_count()) w128 = false;
  auto roles = [&]() -> const char* {
    auto one = [&]() -> const char* {
      if (r128 && w128) return launch_scan_roles_t<128, 128>(a, BH, stream);
      if (r128) return launch_scan_roles_t<128, 64>(a, BH, stream);
      if (w128) return launch_scan_roles_t<64, 128>(a, BH, stream);
      return launch_scan_roles_t<64, 64>(a, BH, stream);
    };
    if (a.nseg > 1) {
      a.seg_phase = 1;
      if (const char* e = one()) return e;
      a.seg_phase = 2;
    }
    return one();
  };
  if (hilo) {
    // Forward that returns the last state: the chunks whose rounding no longer shows in it need no remainder operand.
    // Where the rest are few they run twice in the same kernel; otherwise it leaves its state in final_out / n_final and
    // the kernel with both operands continues from there.  The number is known on the device only (it follows from the
    // decay factors): the second launch is made in any case and ends at once where it has nothing to do, except where late
    // chunks always run twice, and for the sigmoid gate, where all chunks carry the remainder.
    if (a.final_out == nullptr || a.backward) return "scan: the remainder split serves the forward last state only";
    const bool two = a.nstates == nullptr || a.n_final != nullptr;  // n needs its hand-over buffer too
    if (a.repeat_all || (two && !a.all_remainder)) {
      a.part = 1;
      if (const char* e = roles()) return e;
      if (a.repeat_all) return nullptr;
      a.part = 2;
    }
    if (r128 && w128) return launch_scan_t<128, 128, true>(a, BH, stream);
    if (r128) return launch_scan_t<128, 64, true>(a, BH, stream);
    if (w128) return launch_scan_t<64, 128, true>(a, BH, stream);
    return launch_scan_t<64, 64, true>(a, BH, stream);
  }
  return roles();
}

}  // namespace mlstm
