// Native host path of the torch operators: argument checks, output and workspace allocation, the autograd node and the
// calls into libmlstm_hip.so, as a CPython extension module (mlstm_kernels_amd/_torch_host).
//
// What bounds the small calls (one decode step, a short prompt, a toy training step) is the time the host takes to issue
// them, not the kernels: a step kernel of 7 us went out every 25 us when each tensor passed through a dozen Python calls
// and a ctypes marshalling, and the backward of a Python autograd.Function ran its own Python code on the engine's
// thread.  Here a call parses its arguments once (METH_FASTCALL, no keyword handling), allocates through the caching
// allocator and launches; the backward is a C++ autograd node, which needs neither the interpreter nor its lock.
//
// Measured on MI355X, host time to issue one call before / after (all of it Python and ctypes / this module behind the
// same Python operators): decode step through mLSTMBackend 26 / 10 us, 16-token sequence 20 / 7 us, prefill 60 / 20 us,
// forward + backward of B = 1, NH = 4, S = 256 196 / 106 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/mlstm_hip.h"

namespace {

using at::Tensor;

int dtype_code(at::ScalarType t) {  // -1: not a type the kernels take
  switch (t) {
    case at::kFloat: return MLSTM_F32;
    case at::kBFloat16: return MLSTM_BF16;
    case at::kHalf: return MLSTM_F16;
    default: return -1;
  }
}
at::ScalarType scalar_type(int code) {
  return code == MLSTM_F32 ? at::kFloat : (code == MLSTM_BF16 ? at::kBFloat16 : at::kHalf);
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return (float*)ptr(t); }
void* stream_of(const c10::Device& dev) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}
Tensor empty(at::IntArrayRef sizes, at::ScalarType t, const c10::Device& dev) {
  return at::empty(sizes, at::TensorOptions().dtype(t).device(dev));
}
Tensor as_dense(const Tensor& t, at::ScalarType type) {  // t.to(type).contiguous(), without the calls where it is both already
  if (t.scalar_type() == type && t.is_contiguous()) return t;
  return t.to(type).contiguous();
}
void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed: ", mlstm_hip_last_error());
}

// ------------------------------------------------------------------------------------------------ argument parsing
bool is_tensor(PyObject* o) { return THPVariable_Check(o); }
// a tensor, or an undefined one for None
bool opt_tensor(PyObject* o, Tensor& out) {
  if (o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  out = THPVariable_Unpack(o);
  return true;
}
PyObject* wrap_or_none(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject* triple(const Tensor& a, const Tensor& b, const Tensor& c) {
  PyObject* st = PyTuple_New(3);
  PyTuple_SET_ITEM(st, 0, wrap_or_none(a));
  PyTuple_SET_ITEM(st, 1, wrap_or_none(b));
  PyTuple_SET_ITEM(st, 2, wrap_or_none(c));
  return st;
}
PyObject* with_states(const Tensor& h, const Tensor& a, const Tensor& b, const Tensor& c) {
  PyObject* out = PyTuple_New(2);
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(h));
  PyTuple_SET_ITEM(out, 1, triple(a, b, c));
  return out;
}
PyObject* bad_args(const char* what) {
  PyErr_SetString(PyExc_TypeError, what);
  return nullptr;
}

bool same_device(const c10::Device& dev, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->device() != dev) return false;
  return true;
}
bool shape_is(const Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}
bool shape_is(const Tensor& t, int64_t a, int64_t b, int64_t c, int64_t d) {
  return t.dim() == 4 && t.size(0) == a && t.size(1) == b && t.size(2) == c && t.size(3) == d;
}
bool dense(std::initializer_list<const Tensor*> ts, at::ScalarType type) {
  for (const Tensor* t : ts)
    if (t->scalar_type() != type || !t->is_contiguous()) return false;
  return true;
}

// ------------------------------------------------------------------------------------------------ decode step
// step(c, n, m, q, k, v, i, f, c_new, n_new, m_new, eps, state_dtype) -> (h, (c', n', m')), or None when an argument is
// not as the kernel needs it (the caller then converts or names the fault).  q, k, v are (B, NH, D) or (B, NH, 1, D); h
// has v's shape.
PyObject* py_step(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 13) return bad_args("step takes 13 arguments");
  for (int x = 0; x < 8; ++x)
    if (!is_tensor(a[x])) Py_RETURN_NONE;
  const Tensor &c = THPVariable_Unpack(a[0]), &n = THPVariable_Unpack(a[1]), &m = THPVariable_Unpack(a[2]);
  const Tensor &q = THPVariable_Unpack(a[3]), &k = THPVariable_Unpack(a[4]), &v = THPVariable_Unpack(a[5]);
  const Tensor &i = THPVariable_Unpack(a[6]), &f = THPVariable_Unpack(a[7]);
  const double eps = PyFloat_AsDouble(a[11]);
  const int sdt = (int)PyLong_AsLong(a[12]);
  if (PyErr_Occurred()) return nullptr;
  const c10::Device dev = q.device();
  if (!dev.is_cuda() || !same_device(dev, {&c, &n, &m, &k, &v, &i, &f})) Py_RETURN_NONE;
  const at::ScalarType st = scalar_type(sdt);
  const int qdt = dtype_code(q.scalar_type()), gdt = dtype_code(i.scalar_type());
  if (qdt < 0 || gdt < 0 || !dense({&q, &k, &v}, q.scalar_type()) || !dense({&i, &f}, i.scalar_type()) || !dense({&c, &n, &m}, st))
    Py_RETURN_NONE;
  const int64_t d = q.dim();
  if ((d != 3 && !(d == 4 && q.size(2) == 1)) || v.dim() != d) Py_RETURN_NONE;
  const int64_t B = q.size(0), NH = q.size(1), DQ = q.size(d - 1), DV = v.size(d - 1);
  if (d == 3) {
    if (!shape_is(k, B, NH, DQ) || !shape_is(v, B, NH, DV)) Py_RETURN_NONE;
  } else if (!shape_is(k, B, NH, 1, DQ) || !shape_is(v, B, NH, 1, DV)) {
    Py_RETURN_NONE;
  }
  if (!shape_is(c, B, NH, DQ, DV) || !shape_is(n, B, NH, DQ) || !shape_is(m, B, NH, 1) || !shape_is(i, B, NH, 1) ||
      !shape_is(f, B, NH, 1))
    Py_RETURN_NONE;
  Tensor c_new, n_new, m_new;
  if (!opt_tensor(a[8], c_new) || !opt_tensor(a[9], n_new) || !opt_tensor(a[10], m_new)) Py_RETURN_NONE;
  if (c_new.defined() != n_new.defined() || c_new.defined() != m_new.defined()) Py_RETURN_NONE;
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  c10::OptionalDeviceGuard guard(dev);
  if (c_new.defined()) {
    if (!dense({&c_new, &n_new, &m_new}, st) || !same_device(dev, {&c_new, &n_new, &m_new}) || c_new.sizes() != c.sizes() ||
        n_new.sizes() != n.sizes() || m_new.sizes() != m.sizes())
      Py_RETURN_NONE;
  } else {
    c_new = empty(c.sizes(), st, dev);
    n_new = empty(n.sizes(), st, dev);
    m_new = empty(m.sizes(), st, dev);
  }
  const Tensor h = empty(v.sizes(), v.scalar_type(), dev);
  check_rc(mlstm_hip_step(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr(c), ptr(n), ptr(m), ptr(h), ptr(c_new), ptr(n_new),
                          ptr(m_new), (int)B, (int)NH, (int)DQ, (int)DV, (float)eps, qdt, gdt, sdt, stream_of(dev)),
           "mlstm_hip_step");
  return with_states(h, c_new, n_new, m_new);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ multi-token sequence
// sequence(q, k, v, i, f, c, n, m, eps, state_dtype) -> (H, (c', n', m')); the arguments have been checked and converted
// by the caller (dense tensors of one device; q, k, v of one type, i, f of one type, c, n, m of the state type).
PyObject* py_sequence(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 10) return bad_args("sequence takes 10 arguments");
  for (int x = 0; x < 8; ++x)
    if (!is_tensor(a[x])) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  const Tensor &i = THPVariable_Unpack(a[3]), &f = THPVariable_Unpack(a[4]);
  const Tensor &c = THPVariable_Unpack(a[5]), &n = THPVariable_Unpack(a[6]), &m = THPVariable_Unpack(a[7]);
  const double eps = PyFloat_AsDouble(a[8]);
  const int sdt = (int)PyLong_AsLong(a[9]);
  if (PyErr_Occurred()) return nullptr;
  const c10::Device dev = q.device();
  if (!dev.is_cuda() || !same_device(dev, {&k, &v, &i, &f, &c, &n, &m})) Py_RETURN_NONE;
  const at::ScalarType st = scalar_type(sdt);
  const int qdt = dtype_code(q.scalar_type()), gdt = dtype_code(i.scalar_type());
  if (qdt < 0 || gdt < 0 || !dense({&q, &k, &v}, q.scalar_type()) || !dense({&i, &f}, i.scalar_type()) || !dense({&c, &n, &m}, st))
    Py_RETURN_NONE;
  if (q.dim() != 4 || v.dim() != 4) Py_RETURN_NONE;
  const int64_t B = q.size(0), NH = q.size(1), S = q.size(2), DQ = q.size(3), DV = v.size(3);
  if (S == 0 || !shape_is(k, B, NH, S, DQ) || !shape_is(v, B, NH, S, DV) || !shape_is(i, B, NH, S) || !shape_is(f, B, NH, S) ||
      !shape_is(c, B, NH, DQ, DV) || !shape_is(n, B, NH, DQ) || !shape_is(m, B, NH, 1))
    Py_RETURN_NONE;
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  c10::OptionalDeviceGuard guard(dev);
  const Tensor H = empty(v.sizes(), v.scalar_type(), dev);
  const Tensor c_new = empty(c.sizes(), st, dev), n_new = empty(n.sizes(), st, dev), m_new = empty(m.sizes(), st, dev);
  check_rc(mlstm_hip_recurrent_sequence(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr(c), ptr(n), ptr(m), ptr(H), ptr(c_new),
                                        ptr(n_new), ptr(m_new), (int)B, (int)NH, (int)S, (int)DQ, (int)DV, (float)eps, qdt,
                                        gdt, sdt, stream_of(dev)),
           "mlstm_hip_recurrent_sequence");
  return with_states(H, c_new, n_new, m_new);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ chunkwise operator
struct ChunkwiseConfig : torch::CustomClassHolder {
  double eps = 1e-6, norm_eps = 1e-6;
  at::ScalarType autocast_dtype = at::kFloat;
  bool want_last = false, siging = false, normalize = true, recompute = false, f32_as_f16 = false, needs_bw = false;
  int path = 0, stride = 0, norm = 0;
  // for the backward: types of the inputs' gradients
  at::ScalarType qt, kt, vt, it, ft, c0t;
  bool has_c0 = false, has_n0 = false, has_m0 = false;
};

struct Operands {  // what the kernels read: dense, q/k/v in the operand format, states in fp32
  Tensor q, k, v, i, f, c0, n0, m0;
};

Operands prepare(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& i, const Tensor& f, const Tensor& c0,
                 const Tensor& n0, const Tensor& m0, bool siging, bool f32_as_f16) {
  Operands o;
  const at::ScalarType kd =
      q.scalar_type() == at::kHalf || (q.scalar_type() == at::kFloat && f32_as_f16) ? at::kHalf : at::kBFloat16;
  o.q = as_dense(q, kd);
  o.k = as_dense(k, kd);
  o.v = as_dense(v, kd);
  const bool g16 = i.scalar_type() == f.scalar_type() && (i.scalar_type() == at::kBFloat16 || i.scalar_type() == at::kHalf);
  const at::ScalarType gd = g16 ? i.scalar_type() : at::kFloat;
  o.i = as_dense(i, gd);
  o.f = as_dense(f, gd);
  if (c0.defined()) {
    o.c0 = as_dense(c0, at::kFloat);
    o.n0 = as_dense(n0, at::kFloat);
    if (!siging && m0.defined()) o.m0 = as_dense(m0, at::kFloat).reshape({q.size(0), q.size(1)}).contiguous();
  }
  return o;
}

struct Forward {
  Tensor H, c_last, n_last, m_last, ws, rstd;
};

Forward forward_launch(const Operands& o, const ChunkwiseConfig& cfg, const Tensor& n_out, const Tensor& m_out) {
  const int B = (int)o.q.size(0), NH = (int)o.q.size(1), S = (int)o.q.size(2), DQ = (int)o.q.size(3), DV = (int)o.v.size(3);
  const c10::Device dev = o.q.device();
  TORCH_CHECK(cfg.path != MLSTM_PATH_FUSED || o.q.scalar_type() == at::kBFloat16,
              "the fused kernel path supports bfloat16 operands only, got torch.", o.q.scalar_type() == at::kHalf ? "float16" : "float32");
  const size_t ws_bytes = mlstm_hip_chunkwise_fw_workspace_bytes(B, NH, S, DQ, DV, cfg.needs_bw, cfg.path, cfg.stride);
  if (ws_bytes == 0) {
    TORCH_CHECK(!(DQ % 64 == 0 && DQ > 896), "DHQK too large for the HIP chunkwise kernels: ", DQ, " (at most 896)");
    TORCH_CHECK(!(cfg.path == MLSTM_PATH_FUSED && DQ != 128 && DQ != 256 && DQ % 64 == 0 && DV % 64 == 0),
                "the fused kernel path supports DHQK = 128 or 256 only, got ", DQ);
    TORCH_CHECK_VALUE(false, "unsupported shape for the HIP chunkwise kernels: B=", B, ", NH=", NH, ", S=", S, ", DHQK=", DQ,
                      ", DHHV=", DV, " (head dimensions must be multiples of 64, DHQK <= 896, B*NH <= 65535)");
  }
  Forward r;
  Tensor mean;
  if (cfg.norm != MLSTM_NORM_NONE) {
    TORCH_CHECK_VALUE(DV == 64 || DV == 128 || DV == 256 || DV == 512,
                      "the fused head norm needs DHHV = 64, 128, 256 or 512, got ", DV);
    mean = empty({B, NH, S}, at::kFloat, dev);
    r.rstd = empty({B, NH, S}, at::kFloat, dev);
  }
  r.ws = empty({(int64_t)ws_bytes}, at::kByte, dev);
  r.H = empty({B, NH, S, DV}, o.q.scalar_type(), dev);
  if (cfg.want_last) {
    r.c_last = empty({B, NH, DQ, DV}, at::kFloat, dev);
    r.n_last = empty({B, NH, DQ}, at::kFloat, dev);
    r.m_last = empty({B, NH, 1}, at::kFloat, dev);
  }
  check_rc(mlstm_hip_chunkwise_fw(ptr(o.q), ptr(o.k), ptr(o.v), ptr(o.i), ptr(o.f), fptr(o.c0), fptr(o.n0), fptr(o.m0),
                                  ptr(r.H), fptr(n_out), fptr(m_out), fptr(r.c_last), fptr(r.n_last), fptr(r.m_last),
                                  ptr(r.ws), ws_bytes, cfg.needs_bw, B, NH, S, DQ, DV, (float)cfg.eps,
                                  dtype_code(o.q.scalar_type()), dtype_code(o.i.scalar_type()),
                                  cfg.siging ? MLSTM_GATE_SIG : MLSTM_GATE_EXP, cfg.normalize, cfg.path, cfg.stride, cfg.norm,
                                  (float)cfg.norm_eps, fptr(mean), fptr(r.rstd), stream_of(dev)),
           "mlstm_hip_chunkwise_fw");
  return r;
}

// What torch.amp.custom_fwd(cast_inputs=...) does to the arguments under autocast.
Tensor autocast_input(const Tensor& t, const ChunkwiseConfig& cfg) {
  if (!t.defined() || !t.is_floating_point() || !t.is_cuda() || t.scalar_type() == at::kDouble) return t;
  return t.to(cfg.autocast_dtype);
}

class ChunkwiseFunction : public torch::autograd::Function<ChunkwiseFunction> {
 public:
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, Tensor q, Tensor k, Tensor v, Tensor i,
                                                Tensor f, const std::optional<Tensor>& c0_, const std::optional<Tensor>& n0_,
                                                const std::optional<Tensor>& m0_, c10::intrusive_ptr<ChunkwiseConfig> cfg) {
    Tensor c0 = c0_.value_or(Tensor()), n0 = n0_.value_or(Tensor()), m0 = m0_.value_or(Tensor());
    // outputs nobody differentiates (the last states in most losses) arrive undefined in backward instead of as freshly
    // allocated zero tensors the size of the state
    if (ctx) ctx->set_materialize_grads(false);
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    c10::OptionalDeviceGuard guard(q.device());
    if (at::autocast::is_autocast_enabled(at::kCUDA)) {
      for (Tensor* t : {&q, &k, &v, &i, &f, &c0, &n0, &m0}) *t = autocast_input(*t, *cfg);
    }
    const Operands o = prepare(q, k, v, i, f, c0, n0, m0, cfg->siging, cfg->f32_as_f16);
    Forward r = forward_launch(o, *cfg, Tensor(), Tensor());
    if (ctx) {
      Tensor ws = r.ws, c0s;
      if (cfg->recompute) {
        // keep only what lies in front of the chunk states (gate vectors, normaliser states, row normalisers); the
        // backward runs the state scan again, from the initial state when there is one
        const int64_t keep = (int64_t)mlstm_hip_chunkwise_fw_saved_bytes((int)o.q.size(0), (int)o.q.size(1), (int)o.q.size(2),
                                                                         (int)o.q.size(3), (int)o.v.size(3));
        if (ws.numel() > keep) ws = ws.slice(0, 0, keep).clone();
        c0s = o.c0;
      }
      // (with a head norm the normalised rows are what the backward of the norm reads; the others were never stored)
      const bool normed = cfg->norm != MLSTM_NORM_NONE;
      ctx->save_for_backward({o.q, o.k, o.v, o.i, o.f, ws, c0s, normed ? r.H : Tensor(), normed ? r.rstd : Tensor()});
      cfg->qt = q.scalar_type(); cfg->kt = k.scalar_type(); cfg->vt = v.scalar_type();
      cfg->it = i.scalar_type(); cfg->ft = f.scalar_type();
      cfg->has_c0 = c0.defined(); cfg->has_n0 = n0.defined(); cfg->has_m0 = m0.defined();
      cfg->c0t = cfg->has_c0 ? c0.scalar_type() : at::kFloat;
      ctx->saved_data["cfg"] = c10::IValue::make_capsule(cfg);
    }
    if (q.scalar_type() != r.H.scalar_type()) r.H = r.H.to(q.scalar_type());
    if (!cfg->want_last) return {r.H};
    return {r.H, r.c_last, r.n_last, r.m_last};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto cfg = c10::static_intrusive_pointer_cast<ChunkwiseConfig>(ctx->saved_data["cfg"].toCapsule());
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &i = saved[3], &f = saved[4], &c0s = saved[6];
    Tensor ws = saved[5];
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    const c10::Device dev = q.device();
    c10::OptionalDeviceGuard guard(dev);
    const int B = (int)q.size(0), NH = (int)q.size(1), S = (int)q.size(2), DQ = (int)q.size(3), DV = (int)v.size(3);
    const at::ScalarType kd = q.scalar_type();
    void* const stream = stream_of(dev);
    const size_t bw_bytes = mlstm_hip_chunkwise_bw_workspace_bytes(B, NH, S, DQ, DV, cfg->stride);
    const Tensor bws = empty({(int64_t)bw_bytes}, at::kByte, dev), dV = empty(v.sizes(), kd, dev);
    if (cfg->recompute) {
      const size_t full_bytes = mlstm_hip_chunkwise_fw_workspace_bytes(B, NH, S, DQ, DV, 1, cfg->path, cfg->stride);
      Tensor full = empty({(int64_t)full_bytes}, at::kByte, dev);
      full.slice(0, 0, ws.numel()).copy_(ws);
      // dV is not written yet: it holds the states between the segments, as H did in the forward (on that path)
      const bool segments = cfg->path == MLSTM_PATH_AUTO;
      check_rc(mlstm_hip_chunkwise_recompute_states_scratch(ptr(k), ptr(v), fptr(c0s), ptr(full), full_bytes,
                                                            segments ? ptr(dV) : nullptr, segments ? dV.nbytes() : 0, B, NH, S,
                                                            DQ, DV, dtype_code(kd), cfg->stride, stream),
               "mlstm_hip_chunkwise_recompute_states");
      ws = full;
    }
    Tensor dH = grads[0];
    if (!dH.defined()) dH = at::zeros({B, NH, S, DV}, q.options());  // only the last states are differentiated
    dH = as_dense(dH, kd);
    if (saved[8].defined()) {
      // gradient of the normalised rows -> gradient of H
      const Tensor raw = at::empty_like(dH);
      check_rc(mlstm_hip_head_norm_bw(ptr(dH), ptr(saved[7]), fptr(saved[8]), ptr(raw), (size_t)B * NH * S, DV, cfg->norm,
                                      dtype_code(kd), stream),
               "mlstm_hip_head_norm_bw");
      dH = raw;
    }
    Tensor dCl;
    if (grads.size() > 1 && grads[1].defined()) dCl = as_dense(grads[1], at::kFloat);
    const Tensor dQ = empty(q.sizes(), kd, dev), dK = empty(k.sizes(), kd, dev);
    // (gradients of 16-bit gates are rounded where they are summed; gates of two types are left to the conversions below)
    const at::ScalarType gd = cfg->it == cfg->ft && dtype_code(cfg->it) >= 0 ? cfg->it : at::kFloat;
    const Tensor dI = empty({B, NH, S}, gd, dev), dF = empty({B, NH, S}, gd, dev);
    Tensor dC0;
    if (cfg->has_c0) dC0 = empty({B, NH, DQ, DV}, at::kFloat, dev);
    check_rc(mlstm_hip_chunkwise_bw_typed(ptr(q), ptr(k), ptr(v), ptr(i), ptr(f), ptr(dH), fptr(dCl), ptr(dQ), ptr(dK), ptr(dV),
                                          ptr(dI), ptr(dF), fptr(dC0), ptr(ws), (size_t)ws.numel(), ptr(bws), bw_bytes, B, NH, S,
                                          DQ, DV, (float)cfg->eps, dtype_code(kd), dtype_code(i.scalar_type()), dtype_code(gd),
                                          cfg->siging ? MLSTM_GATE_SIG : MLSTM_GATE_EXP, cfg->normalize, cfg->path, cfg->stride,
                                          stream),
             "mlstm_hip_chunkwise_bw");
    Tensor dn0, dm0;
    if (cfg->has_n0) dn0 = at::zeros({B, NH, DQ}, at::TensorOptions().dtype(at::kFloat).device(dev));
    if (cfg->has_m0) dm0 = at::zeros({B, NH, 1}, at::TensorOptions().dtype(at::kFloat).device(dev));
    return {dQ.to(cfg->qt), dK.to(cfg->kt), dV.to(cfg->vt), dI.to(cfg->it), dF.to(cfg->ft),
            dC0.defined() ? dC0.to(cfg->c0t) : dC0, dn0, dm0, Tensor()};
  }
};

bool assert_that(bool ok, const char* what) {
  if (!ok) PyErr_SetString(PyExc_AssertionError, what);
  return ok;
}

// chunkwise(q, k, v, i, f, c0, n0, m0, return_last, eps, autocast_dtype, siging, normalize, path, stride, norm, norm_eps,
//           recompute, float32_as_float16) -> (H, c_last, n_last, m_last), the states None unless asked for
PyObject* py_chunkwise(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 19) return bad_args("chunkwise takes 19 arguments");
  for (int x = 0; x < 5; ++x)
    if (!is_tensor(a[x])) return bad_args("q, k, v, i and f must be tensors");
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  const Tensor &i = THPVariable_Unpack(a[3]), &f = THPVariable_Unpack(a[4]);
  Tensor c0, n0, m0;
  if (!opt_tensor(a[5], c0) || !opt_tensor(a[6], n0) || !opt_tensor(a[7], m0))
    return bad_args("initial states must be tensors or None");
  auto cfg = c10::make_intrusive<ChunkwiseConfig>();
  const int want_last = PyObject_IsTrue(a[8]);
  cfg->want_last = want_last > 0;
  cfg->eps = PyFloat_AsDouble(a[9]);
  cfg->autocast_dtype = scalar_type((int)PyLong_AsLong(a[10]));
  cfg->siging = PyObject_IsTrue(a[11]) > 0;
  cfg->normalize = PyObject_IsTrue(a[12]) > 0;
  cfg->path = (int)PyLong_AsLong(a[13]);
  cfg->stride = (int)PyLong_AsLong(a[14]);
  cfg->norm = (int)PyLong_AsLong(a[15]);
  cfg->norm_eps = PyFloat_AsDouble(a[16]);
  cfg->recompute = PyObject_IsTrue(a[17]) > 0;
  cfg->f32_as_f16 = PyObject_IsTrue(a[18]) > 0;
  if (PyErr_Occurred()) return nullptr;
  TORCH_CHECK(q.is_cuda(), "the 'hip' mLSTM kernels run on an AMD GPU only (got a tensor on '", q.device().str(),
              "'); there is no CPU fallback in mlstm_kernels_amd");
  TORCH_CHECK(same_device(q.device(), {&k, &v, &i, &f}), "all tensors must be on the same device");
  if (!assert_that(q.dim() == 4, "q must have shape (B, NH, S, DHQK)")) return nullptr;
  const int64_t B = q.size(0), NH = q.size(1), S = q.size(2);
  if (!assert_that(k.sizes() == q.sizes(), "k has wrong shape") ||
      !assert_that(v.dim() == 4 && v.size(0) == B && v.size(1) == NH && v.size(2) == S, "v has wrong shape") ||
      !assert_that(shape_is(i, B, NH, S) && shape_is(f, B, NH, S), "i and f must have shape (B, NH, S)"))
    return nullptr;
  if (c0.defined()) {
    if (!assert_that(n0.defined() && (cfg->siging || m0.defined()), "Initial states must be provided together.")) return nullptr;
  }
  bool grad = false;
  if (at::GradMode::is_enabled()) {
    for (const Tensor* t : {&q, &k, &v, &i, &f, (const Tensor*)&c0}) grad = grad || (t->defined() && t->requires_grad());
  }
  cfg->needs_bw = grad;
  // forward-mode tangents go through the node as well, which refuses them: they would be dropped without a word otherwise
  bool tangents = false;
  for (const Tensor* t : {&q, &k, &v, &i, &f, (const Tensor*)&c0, (const Tensor*)&n0, (const Tensor*)&m0})
    tangents = tangents || (t->defined() && t->_fw_grad(/*level=*/0).defined());
  const auto opt = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  torch::autograd::variable_list out;
  {
    pybind11::gil_scoped_release no_gil;
    // without a gradient to keep anything for there is no node to build
    out = grad || tangents ? ChunkwiseFunction::apply(q, k, v, i, f, opt(c0), opt(n0), opt(m0), cfg)
                           : ChunkwiseFunction::forward(nullptr, q, k, v, i, f, opt(c0), opt(n0), opt(m0), cfg);
  }
  PyObject* tup = PyTuple_New(4);
  for (size_t x = 0; x < 4; ++x) PyTuple_SET_ITEM(tup, x, x < out.size() ? wrap_or_none(out[x]) : wrap_or_none(Tensor()));
  return tup;
  END_HANDLE_TH_ERRORS
}

// forward(q, k, v, i, f, c0, n0, m0, eps, siging, normalize, want_last, keep, path, stride, norm, norm_eps, n_out, m_out)
// -> (H, c_last, n_last, m_last, workspace, norm_rstd): one forward launch on operands that are already what the kernels read
PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 19) return bad_args("forward takes 19 arguments");
  Operands o;
  Tensor n_out, m_out;
  Tensor* dst[8] = {&o.q, &o.k, &o.v, &o.i, &o.f, &o.c0, &o.n0, &o.m0};
  for (int x = 0; x < 8; ++x)
    if (!opt_tensor(a[x], *dst[x])) return bad_args("forward takes tensors");
  if (!opt_tensor(a[17], n_out) || !opt_tensor(a[18], m_out)) return bad_args("forward takes tensors");
  ChunkwiseConfig cfg;
  cfg.eps = PyFloat_AsDouble(a[8]);
  cfg.siging = PyObject_IsTrue(a[9]) > 0;
  cfg.normalize = PyObject_IsTrue(a[10]) > 0;
  cfg.want_last = PyObject_IsTrue(a[11]) > 0;
  cfg.needs_bw = PyObject_IsTrue(a[12]) > 0;
  cfg.path = (int)PyLong_AsLong(a[13]);
  cfg.stride = (int)PyLong_AsLong(a[14]);
  cfg.norm = (int)PyLong_AsLong(a[15]);
  cfg.norm_eps = PyFloat_AsDouble(a[16]);
  if (PyErr_Occurred()) return nullptr;
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  c10::OptionalDeviceGuard guard(o.q.device());
  const Forward r = forward_launch(o, cfg, n_out, m_out);
  PyObject* tup = PyTuple_New(6);
  const Tensor* res[6] = {&r.H, &r.c_last, &r.n_last, &r.m_last, &r.ws, &r.rstd};
  for (int x = 0; x < 6; ++x) PyTuple_SET_ITEM(tup, x, wrap_or_none(*res[x]));
  return tup;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"step", (PyCFunction)(void (*)(void))py_step, METH_FASTCALL, "one decode step"},
    {"sequence", (PyCFunction)(void (*)(void))py_sequence, METH_FASTCALL, "several tokens in one launch"},
    {"chunkwise", (PyCFunction)(void (*)(void))py_chunkwise, METH_FASTCALL, "chunkwise forward with autograd backward"},
    {"forward", (PyCFunction)(void (*)(void))py_forward, METH_FASTCALL, "one chunkwise forward launch"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_host", "Native host path of the mLSTM operators", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};
}  // namespace

PyMODINIT_FUNC PyInit__torch_host(void) { return PyModule_Create(&module); }
