// Host-visible launch interface of the kernel translation units (argument structs + launchers).
// Every launcher validates what its kernel's indexing assumes, enqueues on `stream`, and returns nullptr
// on success or a static message describing the rejected argument.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "layout.h"

namespace mlstm {

// Properties of a device that every launch needs and that cost the host about as much as a launch to ask the runtime
// for: kept per device after the first question.
constexpr int kMaxHostDevices = 64;
inline int current_device() {
  int dev = -1;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxHostDevices ? dev : -1;
}
inline int device_cu_count() {
  static std::atomic<int> cached[kMaxHostDevices];
  const int dev = current_device();
  if (dev < 0) return 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}
// The dynamic LDS limit of one kernel (one object per kernel instantiation): raised when a launch needs more than any
// launch on that device before it.  Raising it is one step with recording it: of two threads with different needs the
// one with the smaller could otherwise set the limit last and the larger be recorded as allowed for good.
struct LdsLimit {
  std::atomic<int> bytes[kMaxHostDevices];
  std::mutex raise;
  bool allow(const void* kernel, size_t need) {
    const int dev = current_device();
    if (dev < 0) return false;
    if (bytes[dev].load(std::memory_order_acquire) >= (int)need) return true;
    std::lock_guard<std::mutex> lock(raise);
    if (bytes[dev].load(std::memory_order_relaxed) >= (int)need) return true;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)need) != hipSuccess) return false;
    bytes[dev].store((int)need, std::memory_order_release);
    return true;
  }
};

struct ScanArgs {
  const uint16_t* X;      // (B,NH,S,DHQK) bf16/fp16: K (forward) or Q (backward)
  const uint16_t* Y;      // (B,NH,S,DHHV) bf16/fp16: V (forward) or dH (backward)
  const float* scale_a;   // [BH][Sp] forward: abar; backward: bbar
  const float* nrow;      // backward: [BH][Sp] row normaliser or nullptr; forward: nullptr
  const float* gbar;      // [BH][NC]
  const float* init;      // (B,NH,DHQK,DHHV) fp32 or nullptr (zeros)
  uint16_t* states;       // bf16 fragments [BH][ceil(NC/stride)][DHHV/32][DHQK/16][64][8]
  float* final_out;       // (B,NH,DHQK,DHHV) fp32 or nullptr
  const float* n_init;    // forward: (B,NH,DHQK) or nullptr
  float* nstates;         // forward: [BH][NC][3][DHQK] (three partial vectors per chunk) or nullptr (skip the n recurrence)
  float* n_final;         // forward: (B,NH,DHQK) or nullptr
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int backward;
  int stride;             // a chunk state is kept every `stride` chunks
  int f16;                // X, Y and the state fragments are float16 instead of bfloat16
  int all_remainder;      // forward, last state returned: every chunk carries the remainder of the value operand (the
                          // sigmoid input gate has no stabiliser, so the decay factors alone do not say which chunks
                          // still weigh in the last state)
  float* seg;             // scratch for the states between segments, of seg_bytes (an output that is written later), or nullptr
  size_t seg_bytes;
  int skip_zero;          // the readers of `states` know that the one at the start is zero (init = nullptr): it is not written
  // set by the launcher:
  int n_jobs;             // state tiles * batch * heads * segments
  int end_c, end_n;       // chunks run for the state (in scan order) and for n
  int part;               // 0 whole sequence; 1 / 2 the two launches of a forward scan that returns the last state
  int n_bh;               // batch * heads
  int by_batch;           // the kernels may be chosen by the number of heads (a path that the caller names: not)
  const int* unless;      // device flag, nullptr: none; set: nothing is to be done (whole sequence without the last state only)
  int repeat_all;         // (launch_scan) late chunks always run twice
  int with_backward;      // this is a call with a backward, or the backward
  int nseg, seg_len;      // segments of the sequence, chunks in each (the last one may be shorter)
  int seg_phase;          // 0 one piece; 1 every segment but the last from zero, 2 all segments from their states
};

struct ParHvArgs {
  const uint16_t *Q, *K, *V, *dH;  // forward uses Q,K,V; dV uses Q,K,dH
  GateBufs g;
  const float* nstates;     // forward: n before each chunk, [BH][NC][3][DHQK]: three partial vectors to add up
  const uint16_t* states;   // forward: C states; dV: dC states
  const float* nrow;        // dV: row normaliser (input)
  float* nrow_out;          // forward: row normaliser (output, workspace [BH][Sp])
  uint16_t* Out;            // (B,NH,S,DHHV) bf16: H or dV
  float* n_out;             // forward, optional (B,NH,S)
  float* m_out;             // forward, optional (B,NH,S)
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int sig_gate;
  int use_nrow;             // 0 only for the un-normalised sigmoid-gate variant
  int stride;               // a chunk state is kept every `stride` chunks
  int head_norm;            // forward: 0 none, 1 layer norm, 2 rms norm over the DHHV columns of every row of H
  float norm_eps;
  float* norm_mean;         // forward with head_norm: (B,NH,S) row means (0 for rms)
  float* norm_rstd;         // forward with head_norm: (B,NH,S) reciprocal standard deviations
  int zero_state;           // the state that the first (forward) / last (dV) group of `stride` chunks uses is known to be zero
  int f16;                  // inputs, state fragments and Out are float16 instead of bfloat16
};

struct HeadNormBwArgs {
  const uint16_t* dY;       // (rows, D) bf16 gradient of the normalised output
  const uint16_t* Y;        // (rows, D) bf16 normalised output
  const float* rstd;        // (rows)
  uint16_t* dX;             // (rows, D) bf16 gradient of the input of the norm
  size_t rows;
  int D, kind;              // kind: 1 layer norm, 2 rms norm
  int f16;                  // dY, Y and dX are float16 instead of bfloat16
};

struct FusedHvArgs {
  const uint16_t *Q, *K, *V, *dH;  // forward uses Q,K,V; dV uses Q,K,dH
  GateBufs g;
  const float* init;        // (B,NH,DHQK,DHHV) fp32 initial state (forward: C0, dV: dC_last) or nullptr (zeros)
  const float* n_init;      // forward: (B,NH,DHQK) or nullptr
  const float* nrow;        // dV: row normaliser of the forward pass
  uint16_t* states;         // bf16 state fragments [BH][ceil(NC/stride)][DHHV/32][DHQK/16][64][8] or nullptr (not emitted)
  uint16_t* Out;            // (B,NH,S,DHHV) bf16: H or dV
  float* nrow_out;          // forward: row normaliser (workspace [BH][Sp])
  float* n_out;             // forward, optional (B,NH,S)
  float* m_out;             // forward, optional (B,NH,S)
  float* final_out;         // (B,NH,DHQK,DHHV) fp32 or nullptr: C_last (forward) / dC0 (dV)
  float* n_final;           // forward: (B,NH,DHQK) or nullptr
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int sig_gate;
  int use_nrow;             // 0 only for the un-normalised sigmoid-gate variant (n is then not tracked)
  int stride;               // a chunk state is emitted every `stride` chunks
};

// State recurrence and output in one launch (chain_hv.hip)
struct ChainHvArgs {
  const uint16_t *Q, *K, *V, *dH;  // forward uses Q,K,V; dV uses Q,K,dH
  GateBufs g;
  const float* init;        // (B,NH,DHQK,DHHV) fp32 initial state (forward: C0, dV: dC_last) or nullptr (zeros)
  const float* n_init;      // forward: (B,NH,DHQK) or nullptr
  const float* nrow;        // dV: row normaliser of the forward pass
  uint16_t* states;         // state fragments [BH][ceil(NC/stride)][DHHV/32][DHQK/16][64][8] or nullptr (not kept)
  uint16_t* Out;            // (B,NH,S,DHHV): H or dV
  float* nrow_out;          // forward: row normaliser (workspace [BH][Sp])
  float* n_out;             // forward, optional (B,NH,S)
  float* m_out;             // forward, optional (B,NH,S)
  float* final_out;         // (B,NH,DHQK,DHHV) fp32 or nullptr: C_last (forward) / dC0 (dV)
  float* n_final;           // forward: (B,NH,DHQK) or nullptr
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int sig_gate;
  int use_nrow;             // 0 only for the un-normalised sigmoid-gate variant (n is then not tracked)
  int stride;               // a chunk state is kept every `stride` chunks
  int f16;
  int skip_zero;            // the first kept state is zero and its readers know
};

constexpr int kShortMax = 512;  // longest sequence of the short forward
struct ShortFwArgs {
  const uint16_t *Q, *K, *V;
  int own_gates;            // the workgroups scan the gates themselves; otherwise the vectors of the pre-pass are in g
  GateBufs g;
  const void *ig, *fg;      // own gates: (B,NH,S) pre-activations
  const float* m0;          // own gates: (B,NH) or nullptr (zeros)
  float* m_last;            // own gates: (B,NH) or nullptr; not m0
  uint16_t* Out;            // (B,NH,S,DHHV)
  float* n_out;             // optional (B,NH,S)
  float* m_out;             // optional (B,NH,S)
  const float* init;        // (B,NH,DHQK,DHHV) or nullptr
  const float* n_init;      // (B,NH,DHQK), with init
  float* final_out;         // (B,NH,DHQK,DHHV) fp32 or nullptr
  float* n_final;           // (B,NH,DHQK) or nullptr (also: n is not tracked)
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int sig_gate, use_nrow;
  int f16, dtype_gates;
};

struct ParQkArgs {
  const uint16_t *Q, *K, *V, *dH;
  GateBufs g;
  const uint16_t* states;   // dQ: C states; dK: dC states
  const float* nrow;
  uint16_t* Out;            // (B,NH,S,DHQK) bf16: dQ or dK
  float* rowdot;            // [DHQK tiles][BH][Sp]: sum_d q*dQ (dQ) or sum_d k*dK (dK) over the rows of one tile
  const uint16_t* states2;  // the dK operands (dC states, dK, sum_d k*dK); states, Out and rowdot above are the
  uint16_t* Out2;           // dQ operands
  float* rowdot2;
  int S, NC, DHQK, DHHV;
  float qk_scale, eps;
  int use_nrow;
  int stride;               // a chunk state is kept every `stride` chunks
  int zero_dc;              // the gradient of the state after the last chunk is known to be zero (of the initial state: g.zero_c)
  int f16;                  // inputs, state fragments and outputs are float16 instead of bfloat16
};

struct GateGradArgs {
  const void *i, *f;        // gate pre-activations (B,NH,S)
  const float *qdq, *kdk;   // [ntiles][BH][Sp]: one slot per head-dimension tile of the dQ/dK kernel
  int ntiles;
  void *dI, *dF;            // (B,NH,S)
  int S, NC, dtype_gates, sig_gate;
  int dtype_grads;          // of dI and dF: 0 fp32, 1 bf16, 2 fp16
};

const char* launch_step(const void* q, const void* k, const void* v, const void* i, const void* f,
                        const void* c_in, const void* n_in, const void* m_in, void* h, void* c_out,
                        void* n_out, void* m_out, int B, int NH, int DHQK, int DHHV, float eps,
                        int dtype_qkv, int dtype_gates, int dtype_state, hipStream_t stream);
const char* launch_step_seq(const void* q, const void* k, const void* v, const void* i, const void* f,
                            const void* c_in, const void* n_in, const void* m_in, void* h, void* c_out,
                            void* n_out, void* m_out, int B, int NH, int T, int DHQK, int DHHV, float eps,
                            int dtype_qkv, int dtype_gates, int dtype_state, hipStream_t stream);
// the same recurrence on the matrix cores, tokens in blocks, for the types and shapes it supports
struct StepBlockArgs {
  const void *q, *k, *v, *i, *f, *c_in, *n_in, *m_in;
  void *h, *c_out, *n_out, *m_out;
  int BH, T, DHQK, DHHV;
  float eps;
  int dtype_qkv, dtype_gates, dtype_state;
};
bool step_block_supported(int DHQK, int DHHV, int dtype_qkv);
const char* launch_step_block(const StepBlockArgs& a, hipStream_t stream);
const char* launch_gates(const void* i, const void* f, const float* m0, const GateBufs& gb, float* m_last,
                         int B, int NH, int S, int dtype_gates, int sig_gate, int zero_c, int chained, hipStream_t stream);
const char* launch_scan(const ScanArgs& a, int BH, bool hilo, hipStream_t stream);
const char* launch_par_hv(const ParHvArgs& a, int BH, bool is_dv, hipStream_t stream);
bool par_hv_head_norm_supported(int DHHV);
bool par_hv_group_each(const ParHvArgs& a, int BH);  // whether launch_par_hv has a workgroup and a CU for every column group
// streaming (persistent, producer / consumer waves) form of the same two kernels for the shapes it supports
bool stream_hv_supported(const ParHvArgs& a);
const char* launch_stream_hv(const ParHvArgs& a, int BH, bool is_dv, hipStream_t stream);
// form of the same two kernels for windows of two chunks (state stride 2), any head dimensions
bool window_hv_supported(const ParHvArgs& a);
bool window_hv_preferred(const ParHvArgs& a, int BH);  // supported, and faster than the tiled kernel at this size
const char* launch_window_hv(const ParHvArgs& a, int BH, bool is_dv, hipStream_t stream);
// forward without backward of a short sequence: H and the last state in one launch
bool short_fw_preferred(const ShortFwArgs& a, int BH);
bool short_fw_own_gates(const ShortFwArgs& a, int BH);
const char* launch_short_fw(const ShortFwArgs& a, int BH, hipStream_t stream);
const char* launch_head_norm_bw(const HeadNormBwArgs& a, hipStream_t stream);
bool chain_hv_preferred(const ChainHvArgs& a, int BH);
const char* launch_chain_hv(const ChainHvArgs& a, int BH, bool is_dv, hipStream_t stream);
const char* launch_chain_states(const ChainHvArgs& a, int BH, hipStream_t stream);  // kept states only, if g.chained is set
bool fused_hv_supported(int DHQK, int DHHV);
const char* launch_fused_hv(const FusedHvArgs& a, int BH, bool is_dv, hipStream_t stream);
const char* launch_par_qk_pair(const ParQkArgs& a, int BH, hipStream_t stream);
// streaming (persistent, producer / consumer waves) form of the same launch for windows of two chunks
bool window_qk_supported(const ParQkArgs& a);
bool window_qk_preferred(const ParQkArgs& a, int BH);
const char* launch_window_qk(const ParQkArgs& a, int BH, hipStream_t stream);
int par_qk_head_tile(int DHQK);  // head-dimension rows per workgroup of the dQ/dK kernel
const char* launch_gate_grads(const GateGradArgs& a, int BH, hipStream_t stream);
const char* launch_fill_zero(float* p, size_t n, hipStream_t stream);
// stores `msg` as the calling thread's last error (what mlstm_hip_last_error returns) and returns 1
int set_last_error(const char* msg);

}  // namespace mlstm
