// Eager host path of the public functions: one call from Python does what the interface module otherwise does in a
// dozen steps of its own (checks, outputs and scratch from torch's allocator, argument structs, the library calls, the
// autograd node).  It adds nothing to the device work: everything runs through the C ABI of libflash_moba_hip.so.
//
// Why it exists: a small call (two sequences, 3072 tokens, forward) issues its kernels in about 60 us of device time,
// and the Python host needed 160 us to issue them -- the dispatch of four custom ops, ctypes structs of forty fields,
// a device guard and a stream look-up per op.
//
// Every function returns None when a call is not plain eager work on ordinary tensors (tracing, fake or wrapped
// tensors, dispatch modes) or its arguments are not of the common form (non-contiguous last dimension, a head dimension
// that has to be padded, empty sequences, anything the checks would reject): the caller then takes the path in Python,
// which handles or reports it.
#include <torch/extension.h>

#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <optional>
#include <tuple>
#include <utility>

#include "../../include/flash_moba_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc) {
  if (rc != 0) throw std::runtime_error(fmoba_last_error());
}

// A C++ exception of the base class becomes RuntimeError in Python.  The device check is made once per device.
void check_device(int index) {
  static std::atomic<uint64_t> ok{0};
  const uint64_t bit = uint64_t(1) << (index & 63);
  if (index < 64 && (ok.load(std::memory_order_relaxed) & bit)) return;
  check(fmoba_check_device());
  if (index < 64) ok.fetch_or(bit);
}

PyObject *g_parameter_class = nullptr;  // torch.nn.Parameter

// an ordinary tensor (or parameter): no subclass, no wrapper of a transform, no lazy conjugate, no tangent of forward-mode
// differentiation (a dual tensor has the key set of an ordinary one; the path in Python refuses it, having no derivative of that kind)
bool plain(const py::handle &h) {
  if (!THPVariable_CheckExact(h.ptr()) && reinterpret_cast<PyObject *>(Py_TYPE(h.ptr())) != g_parameter_class) return false;
  const Tensor &t = THPVariable_Unpack(h.ptr());
  return t.defined() && t.is_cuda() && !t.is_sparse() && !t._fw_grad(/*level=*/0).defined() &&
         !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative}));
}

bool eager() { return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing(); }

bool is_cu(const Tensor &t, int64_t n, const at::Device &dev) {
  return t.scalar_type() == at::kInt && t.dim() == 1 && t.numel() == n && t.is_contiguous() && t.device() == dev;
}

// (rows, heads, dim), last dimension dense, 16-byte vectors
bool is_rows(const Tensor &t, at::ScalarType dt, const at::Device &dev) {
  return t.dim() == 3 && t.scalar_type() == dt && t.device() == dev && t.stride(2) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct Shape {
  int64_t total_q, total_k, heads, heads_k, dim, batch, max_q, max_k, chunk, max_cols;
  bool causal;
  int dtype;
  void *stream;
};

// fills `s` and says whether the call is of the common form
bool common_form(Shape &s, const Tensor &q, const Tensor &k, const Tensor &cu_q, const Tensor &cu_k, int64_t max_q, int64_t max_k,
                 int64_t chunk, bool causal) {
  const at::ScalarType dt = q.scalar_type();
  if (dt != at::kHalf && dt != at::kBFloat16) return false;
  const at::Device dev = q.device();
  if (!is_rows(q, dt, dev) || !is_rows(k, dt, dev)) return false;
  s.batch = cu_q.numel() - 1;
  if (s.batch < 1 || s.batch > 65535 || !is_cu(cu_q, s.batch + 1, dev) || !is_cu(cu_k, s.batch + 1, dev)) return false;
  s.total_q = q.size(0), s.total_k = k.size(0), s.heads = q.size(1), s.heads_k = k.size(1), s.dim = q.size(2);
  if (s.total_q < 1 || s.total_k < 1 || s.heads < 1 || s.heads_k < 1 || s.heads % s.heads_k != 0 || s.heads > 65535) return false;
  if (k.size(2) != s.dim || s.dim % 8 != 0 || s.dim < 8 || s.dim > 256) return false;
  if (max_q < 1 || max_k < 1 || chunk < 1 || max_q > INT32_MAX || max_k > INT32_MAX || chunk > INT32_MAX || s.total_q > INT32_MAX || s.total_k > INT32_MAX) return false;
  s.max_q = max_q, s.max_k = max_k, s.chunk = chunk, s.causal = causal;
  s.max_cols = (max_k + chunk - 1) / chunk;
  s.dtype = dt == at::kBFloat16 ? FMOBA_DTYPE_BF16 : FMOBA_DTYPE_F16;
  return true;
}

Tensor bytes_like(const Tensor &q, size_t n) { return at::empty({static_cast<int64_t>(std::max<size_t>(n, 1))}, q.options().dtype(at::kByte)); }
size_t up256(size_t x) { return (x + 255) & ~size_t(255); }

struct Pattern {
  Tensor col_offsets, col_nnz, indices, scratch;
  Tensor visits;                        // defined: the lists are ranked (gated patterns whose attention leaves partial results per visit)
  const uint32_t *selection = nullptr;  // in `scratch`
};

// chunk means, gating and (with `lists`) the column lists, ranked if wanted; `attn`: with the forward that takes the gate's place
Pattern gate(const Shape &s, const Tensor &q, const Tensor &k, const Tensor &cu_q, const Tensor &cu_k, int64_t topk, bool lists, bool ranked = false,
             const fmoba_attn_fwd_args *attn = nullptr) {
  Pattern p;
  const auto i32 = q.options().dtype(at::kInt);
  if (lists) {
    p.col_offsets = at::empty({s.batch, s.heads, s.max_cols}, q.options().dtype(at::kLong));
    p.col_nnz = at::empty({s.batch, s.heads, s.max_cols}, i32);
    p.indices = at::empty({s.total_q * s.heads * topk}, i32);
  }
  // one block of scratch: the gating's workspace (the selection bits at its start), offsets of the pooled sequences, chunk means
  const size_t gate_bytes = up256(fmoba_fused_topk_workspace_bytes(s.batch, s.total_q, s.heads, s.max_q, s.max_k, s.chunk));
  const size_t cu_bytes = up256((s.batch + 1) * 4);
  const size_t km_bytes = static_cast<size_t>(s.total_k / s.chunk + s.batch) * s.heads_k * s.dim * 2;
  const size_t pre_bytes = ranked && s.max_cols > 32 ? up256(static_cast<size_t>(s.heads) * ((s.max_cols + 31) / 32) * s.total_q) : 0;
  p.scratch = bytes_like(q, gate_bytes + cu_bytes + pre_bytes + km_bytes + 256);
  if (ranked) p.visits = at::empty({s.heads, s.total_q}, i32);
  char *base = reinterpret_cast<char *>(up256(reinterpret_cast<size_t>(p.scratch.data_ptr())));
  fmoba_mean_pool_args m{};
  m.k = k.data_ptr(), m.km = base + gate_bytes + cu_bytes + pre_bytes;
  m.cu_seqlens_k = cu_k.data_ptr<int32_t>(), m.cu_seqlens_km = reinterpret_cast<int32_t *>(base + gate_bytes);
  m.batch = s.batch, m.max_chunks = s.max_cols, m.heads_k = s.heads_k, m.head_dim = s.dim, m.chunk = s.chunk, m.dtype = s.dtype;
  m.k_row_stride = k.stride(0), m.k_head_stride = k.stride(1), m.km_row_stride = s.heads_k * s.dim, m.km_head_stride = s.dim;
  fmoba_fused_topk_args g{};
  g.q = q.data_ptr(), g.km = m.km, g.cu_seqlens_q = cu_q.data_ptr<int32_t>(), g.cu_seqlens_k = m.cu_seqlens_k, g.cu_seqlens_km = m.cu_seqlens_km;
  if (lists) g.col_offsets = p.col_offsets.data_ptr<int64_t>(), g.col_nnz = p.col_nnz.data_ptr<int32_t>(), g.flat_indices = p.indices.data_ptr<int32_t>();
  g.workspace = base, g.workspace_bytes = gate_bytes;
  g.batch = s.batch, g.total_q = s.total_q, g.heads = s.heads, g.heads_k = s.heads_k, g.head_dim = s.dim;
  g.max_seqlen_q = s.max_q, g.max_seqlen_k = s.max_k, g.topk = topk, g.chunk = s.chunk, g.is_causal = s.causal, g.dtype = s.dtype;
  g.q_row_stride = q.stride(0), g.q_head_stride = q.stride(1), g.km_row_stride = m.km_row_stride, g.km_head_stride = m.km_head_stride;
  if (attn != nullptr) {
    check(fmoba_attn_fwd_gated_rows(&m, &g, attn, lists ? 1 : 0, s.stream));
  } else if (ranked) {
    const fmoba_csc_ranks r{reinterpret_cast<uint32_t *>(p.visits.data_ptr<int32_t>()), pre_bytes ? reinterpret_cast<uint8_t *>(base + gate_bytes + cu_bytes) : nullptr};
    check(fmoba_pool_and_gate_ranked(&m, &g, &r, s.stream));
  } else {
    check(fmoba_pool_and_gate(&m, &g, lists ? 1 : 0, s.stream));
  }
  p.selection = reinterpret_cast<const uint32_t *>(base);
  return p;
}

fmoba_attn_fwd_args forward_args(const Shape &s, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_q, const Tensor &cu_k,
                                 int64_t visits, double scale, const uint32_t *selection) {
  fmoba_attn_fwd_args a{};
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr();
  a.cu_seqlens_q = cu_q.data_ptr<int32_t>(), a.cu_seqlens_k = cu_k.data_ptr<int32_t>(), a.selection_bits = selection;
  a.batch = s.batch, a.total_q = s.total_q, a.total_k = s.total_k, a.heads = s.heads, a.heads_k = s.heads_k, a.head_dim = s.dim;
  a.max_seqlen_q = s.max_q, a.max_seqlen_k = s.max_k, a.max_cols = s.max_cols, a.lg_block_m = 128, a.lg_block_n = s.chunk;
  a.is_causal = s.causal && s.max_q != 1;  // (one query row per sequence is never masked: flash_moba_api.cpp:450)
  a.dtype = s.dtype, a.max_visits_per_row = visits, a.softmax_scale = static_cast<float>(scale);
  a.q_row_stride = q.stride(0), a.q_head_stride = q.stride(1), a.k_row_stride = k.stride(0), a.k_head_stride = k.stride(1);
  a.v_row_stride = v.stride(0), a.v_head_stride = v.stride(1);
  return a;
}

struct Result {
  Tensor out, lse;
};
const uint32_t *visit_ptr(const Tensor &t) { return t.defined() ? reinterpret_cast<const uint32_t *>(t.data_ptr<int32_t>()) : nullptr; }

// the tensors that a forward writes
Result results(const Shape &s, fmoba_attn_fwd_args &a, const Tensor &q) {
  Result r;
  r.out = at::empty_like(q);
  r.lse = at::empty({s.heads, s.total_q}, q.options().dtype(at::kFloat));
  a.out = r.out.data_ptr(), a.softmax_lse = r.lse.data_ptr<float>();
  a.o_row_stride = r.out.stride(0), a.o_head_stride = r.out.stride(1);
  return r;
}
// what this thread's last forward ran, and its last backward if nobody has asked since (else -1): diagnostics
thread_local int t_visits = 0, t_row_blocks = 0, t_partials = -1;

// gate and attention of a call with a few query rows per sequence
Result forward_few(const Shape &s, fmoba_attn_fwd_args a, const Tensor &q, const Tensor &k, int64_t topk, size_t score_bytes) {
  const Result r = results(s, a, q);
  const size_t cu_bytes = up256((s.batch + 1) * 4);
  const Tensor scratch = bytes_like(q, cu_bytes + score_bytes + 256);
  char *base = reinterpret_cast<char *>(up256(reinterpret_cast<size_t>(scratch.data_ptr())));
  fmoba_mean_pool_args m{};
  m.k = a.k;
  m.cu_seqlens_k = a.cu_seqlens_k, m.cu_seqlens_km = reinterpret_cast<int32_t *>(base);
  m.batch = s.batch, m.max_chunks = s.max_cols, m.heads_k = s.heads_k, m.head_dim = s.dim, m.chunk = s.chunk, m.dtype = s.dtype;
  m.k_row_stride = k.stride(0), m.k_head_stride = k.stride(1);
  t_visits = a.max_visits_per_row, t_row_blocks = 1;
  check(fmoba_attn_fwd_gated_few(&m, &a, topk, s.causal, reinterpret_cast<float *>(base + cu_bytes), s.stream));
  return r;
}

// what the form of dQ and its workspace depend on
void backward_sizes(fmoba_attn_bwd_args &b, const Shape &s, int64_t visits64) {
  b.batch = s.batch, b.total_q = s.total_q, b.total_k = s.total_k, b.heads = s.heads, b.heads_k = s.heads_k, b.head_dim = s.dim;
  b.max_seqlen_q = s.max_q, b.max_seqlen_k = s.max_k, b.max_cols = s.max_cols, b.lg_block_n = s.chunk, b.is_causal = s.causal && s.max_q != 1;
  b.max_visits_per_row = visits64;
}

Result forward(const Shape &s, fmoba_attn_fwd_args a, const Tensor &q, const Pattern &p) {
  const Result r = results(s, a, q);
  if (p.indices.defined()) a.col_offsets = p.col_offsets.data_ptr<int64_t>(), a.col_nnz = p.col_nnz.data_ptr<int32_t>(), a.row_indices = p.indices.data_ptr<int32_t>();
  t_visits = a.max_visits_per_row;
  t_row_blocks = fmoba_attn_fwd_uses_row_blocks(&a);
  const size_t n = fmoba_attn_fwd_workspace_bytes(&a);
  const Tensor ws = bytes_like(q, n);
  a.workspace = ws.data_ptr(), a.workspace_bytes = n;
  check(fmoba_attn_fwd_ranked(&a, visit_ptr(p.visits), 3, s.stream));
  return r;
}

// forward and backward of the attention over a pattern: the node of the autograd graph
struct Attention : public torch::autograd::Function<Attention> {
  // the pattern and the results of the forward pass are made by the caller, below autograd; this records them
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_q, const Tensor &cu_k,
                        const Pattern &p, const Result &r, int64_t max_q, int64_t max_k, int64_t chunk, bool causal, double scale, int64_t bwd_visits,
                        bool deterministic) {
    ctx->save_for_backward({q, k, v, r.out, r.lse, cu_q, cu_k, p.col_offsets, p.col_nnz, p.indices, p.visits});
    ctx->saved_data["max_q"] = max_q;
    ctx->saved_data["max_k"] = max_k;
    ctx->saved_data["chunk"] = chunk;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["visits"] = bwd_visits;
    ctx->saved_data["deterministic"] = deterministic;
    return r.out;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list t = ctx->get_saved_variables();
    const Tensor &q = t[0], &k = t[1], &v = t[2], &out = t[3], &lse = t[4], &cu_q = t[5], &cu_k = t[6], &co = t[7], &cn = t[8], &ind = t[9];
    // What was saved may have been through saved-tensor hooks: nothing of it is taken on trust, as its addresses go to kernels.
    TORCH_CHECK(q.defined() && q.is_cuda(), "flash_moba: a saved tensor is not on the GPU");
    const at::Device dev = q.device();
    const at::ScalarType dt = q.scalar_type();
    for (int i = 0; i < 4; ++i) {
      TORCH_CHECK(t[i].defined() && t[i].device() == dev && t[i].scalar_type() == dt && t[i].dim() == 3, "flash_moba: q, k, v or out was saved and came back as another tensor");
      if (!is_rows(t[i], dt, dev)) t[i] = t[i].contiguous();
    }
    TORCH_CHECK(out.sizes() == q.sizes() && v.sizes() == k.sizes(), "flash_moba: q, k, v or out was saved and came back in another shape");
    const int64_t nb = cu_q.defined() ? cu_q.numel() - 1 : 0;
    auto is = [&](const Tensor &x, at::ScalarType type) { return x.defined() && x.device() == dev && x.scalar_type() == type && x.is_contiguous(); };
    TORCH_CHECK(is(lse, at::kFloat) && lse.dim() == 2 && lse.size(0) == q.size(1) && lse.size(1) == q.size(0) && is(cu_q, at::kInt) && is(cu_k, at::kInt) &&
                    is(co, at::kLong) && is(cn, at::kInt) && is(ind, at::kInt) && co.dim() == 3 && co.sizes() == cn.sizes() && co.size(0) == nb && co.size(1) == q.size(1),
                "flash_moba: the pattern, the offsets or the log-sum-exp was saved and came back as another tensor");
    const Tensor &visits = t[10];
    TORCH_CHECK(!visits.defined() || (is(visits, at::kInt) && visits.numel() == lse.numel()), "flash_moba: the visits of the pattern were saved and came back as another tensor");
    auto num = [&](const char *name) { return ctx->saved_data[name].toInt(); };
    variable_list res(14);  // one per argument of forward
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const c10::DeviceGuard guard(q.device());
      Shape s;
      TORCH_CHECK(common_form(s, q, k, cu_q, cu_k, num("max_q"), num("max_k"), num("chunk"), ctx->saved_data["causal"].toBool()), "flash_moba: saved tensors changed");
      s.stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
      Tensor dout = grads[0];
      TORCH_CHECK(dout.defined() && dout.sizes() == q.sizes() && dout.device() == dev, "flash_moba: no gradient of the shape of the output");
      if (!is_rows(dout, dt, dev)) dout = dout.to(dt).contiguous();
      Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
      fmoba_attn_bwd_args a{};
      a.batch = s.batch, a.total_q = s.total_q, a.total_k = s.total_k, a.heads = s.heads, a.heads_k = s.heads_k, a.head_dim = s.dim;
      a.max_seqlen_q = s.max_q, a.max_seqlen_k = s.max_k, a.max_cols = co.size(2), a.lg_block_m = 128, a.lg_block_n = s.chunk;
      a.is_causal = s.causal && s.max_q != 1, a.dtype = s.dtype, a.deterministic = ctx->saved_data["deterministic"].toBool();
      a.max_visits_per_row = num("visits"), a.softmax_scale = static_cast<float>(ctx->saved_data["scale"].toDouble());
      // heads of a group that the library does not add up itself are summed below (flash_moba_api.cpp:842-845)
      const int32_t dkv_heads = fmoba_attn_bwd_dkv_heads(&a);
      const bool grouped = dkv_heads != s.heads_k;
      const Tensor softmax_d = at::empty({s.heads, s.total_q + 128 * s.batch}, q.options().dtype(at::kFloat));
      a.dout = dout.data_ptr(), a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr(), a.out = out.data_ptr(), a.softmax_lse = lse.data_ptr<float>();
      a.dq = dq.data_ptr(), a.dk = dk.data_ptr(), a.dv = dv.data_ptr(), a.softmax_d = softmax_d.data_ptr<float>();
      a.col_offsets = co.data_ptr<int64_t>(), a.col_nnz = cn.data_ptr<int32_t>(), a.row_indices = ind.data_ptr<int32_t>(), a.num_row_indices = ind.numel();
      a.cu_seqlens_q = cu_q.data_ptr<int32_t>(), a.cu_seqlens_k = cu_k.data_ptr<int32_t>();
      a.q_row_stride = q.stride(0), a.q_head_stride = q.stride(1), a.k_row_stride = k.stride(0), a.k_head_stride = k.stride(1);
      a.v_row_stride = v.stride(0), a.v_head_stride = v.stride(1), a.o_row_stride = out.stride(0), a.o_head_stride = out.stride(1);
      a.do_row_stride = dout.stride(0), a.do_head_stride = dout.stride(1), a.dq_row_stride = dq.stride(0), a.dq_head_stride = dq.stride(1);
      a.dk_row_stride = dk.stride(0), a.dk_head_stride = dk.stride(1), a.dv_row_stride = dv.stride(0), a.dv_head_stride = dv.stride(1);
      const size_t n = fmoba_attn_bwd_workspace_bytes(&a);
      const int64_t one = grouped ? int64_t(s.total_k) * dkv_heads * s.dim : 0;
      const Tensor ws = bytes_like(q, up256(n) + 4 * one);  // the heads kept apart lie behind the library's workspace
      char *apart = static_cast<char *>(ws.data_ptr()) + up256(n);
      if (grouped) {
        a.dk = apart, a.dv = apart + 2 * one;
        a.dk_row_stride = a.dv_row_stride = int64_t(dkv_heads) * s.dim, a.dk_head_stride = a.dv_head_stride = s.dim;
      }
      a.workspace = ws.data_ptr(), a.workspace_bytes = n;
      check(fmoba_attn_bwd_ranked(&a, visit_ptr(visits), dkv_heads, 7, s.stream));
      t_partials = fmoba_attn_bwd_uses_partials(&a);
      if (grouped)
        check(fmoba_sum_grouped_heads(apart, dk.data_ptr(), dv.data_ptr(), s.total_k, dkv_heads, s.heads_k, s.dim, dk.stride(0), dk.stride(1), dv.stride(0), dv.stride(1), s.dtype, s.stream));
      res[0] = dq, res[1] = dk, res[2] = dv;
    }
    if (at::GradMode::is_enabled()) {  // the gradients have no gradients: say so if anything asks for them
      auto error = std::make_shared<torch::autograd::DelayedError>("trying to differentiate twice through flash_moba's backward, which has no derivative", 3);
      for (int i = 0; i < 3; ++i) res[i].requires_grad_(true);
      variable_list wrapped = (*error)({res[0], res[1], res[2]});
      for (int i = 0; i < 3; ++i) res[i] = wrapped[i];
    }
    return res;
  }
};

py::object none() { return py::none(); }

// flash_moba_varlen_func
py::object moba_varlen(const py::handle &hq, const py::handle &hk, const py::handle &hv, const py::handle &hcq, const py::handle &hck, int64_t max_q,
                       int64_t max_k, int64_t chunk, int64_t topk, bool causal) {
  if (!eager() || !plain(hq) || !plain(hk) || !plain(hv) || !plain(hcq) || !plain(hck)) return none();
  const Tensor &q = THPVariable_Unpack(hq.ptr()), &k = THPVariable_Unpack(hk.ptr()), &v = THPVariable_Unpack(hv.ptr());
  const Tensor &cu_q = THPVariable_Unpack(hcq.ptr()), &cu_k = THPVariable_Unpack(hck.ptr());
  Shape s;
  if (!common_form(s, q, k, cu_q, cu_k, max_q, max_k, chunk, causal)) return none();
  if (!is_rows(v, q.scalar_type(), q.device()) || v.sizes() != k.sizes() || chunk % 64 != 0 || topk < 1 || topk > 64) return none();
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  const double scale = std::pow(static_cast<double>(s.dim), -0.5);
  const int kb = fmoba_attn_fwd_key_block(chunk);
  const int64_t visits = topk * (chunk / kb);  // a gated row visits at most top-k chunks
  Tensor out;
  {
    py::gil_scoped_release nogil;
    Pattern p;
    Result r;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const c10::DeviceGuard guard(q.device());
      check_device(q.device().index());
      s.stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
      fmoba_attn_fwd_args a = forward_args(s, q, k, v, cu_q, cu_k, visits, scale, nullptr);
      const size_t few = grad ? 0 : fmoba_attn_fwd_gated_few_bytes(&a);
      if (few > 0) {
        r = forward_few(s, a, q, k, topk, few);
      } else {
        const bool columns = !fmoba_attn_fwd_uses_row_blocks(&a), lists = grad || columns;  // (the row-block form reads the selection bits alone)
        // Ranks for the forms that leave a partial result per visit.  (One query row per sequence: the attention then drops the
        // causal rule that the gating keeps, and the visits of a row are others.  65536 visits: more than a row's count holds.)
        fmoba_attn_bwd_args b{};
        backward_sizes(b, s, visits * (kb / 64));
        const bool ranked = max_q > 1 && visits * (kb / 64) < 65536 && (columns || (grad && fmoba_attn_bwd_uses_partials(&b)));
        if (!ranked && fmoba_attn_fwd_gates_rows(&a)) {
          t_visits = a.max_visits_per_row, t_row_blocks = 1;
          r = results(s, a, q);
          p = gate(s, q, k, cu_q, cu_k, topk, lists, false, &a);
        } else {
          p = gate(s, q, k, cu_q, cu_k, topk, lists, ranked);
          a.selection_bits = p.selection;
          r = forward(s, a, q, p);
        }
      }
    }
    out = grad ? Attention::apply(q, k, v, cu_q, cu_k, p, r, max_q, max_k, chunk, causal, scale, visits * (kb / 64), false) : r.out;
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

// flash_topk_varlen_func
py::object topk_varlen(const py::handle &hq, const py::handle &hk, const py::handle &hcq, const py::handle &hck, int64_t max_q, int64_t max_k,
                       int64_t topk, int64_t chunk, bool causal) {
  if (!eager() || !plain(hq) || !plain(hk) || !plain(hcq) || !plain(hck)) return none();
  const Tensor &q = THPVariable_Unpack(hq.ptr()), &k = THPVariable_Unpack(hk.ptr());
  const Tensor &cu_q = THPVariable_Unpack(hcq.ptr()), &cu_k = THPVariable_Unpack(hck.ptr());
  Shape s;
  if (!common_form(s, q, k, cu_q, cu_k, max_q, max_k, chunk, causal) || topk < 1 || topk > 64) return none();
  Pattern p;
  {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(q.device());
    check_device(q.device().index());
    s.stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
    p = gate(s, q, k, cu_q, cu_k, topk, true);
  }
  return py::make_tuple(p.col_offsets, p.col_nnz, p.indices);
}

// largest number of (row, forward key block) visits of any (row, head): one pass over the lists and a read-back
int64_t count_visits(const fmoba_attn_fwd_args &a, const Tensor &q, void *stream) {
  const int64_t rows = q.size(0) * q.size(1);
  const Tensor counts = at::empty({rows + 1}, q.options().dtype(at::kInt));
  int32_t *c = counts.data_ptr<int32_t>();
  check(fmoba_csc_max_row_visits(&a, c, c + rows, stream));
  return std::max<int64_t>(1, counts.select(0, rows).item<int32_t>());
}

constexpr size_t kUncountedBytes = size_t(8) << 30;

// flash_moba_attn_varlen_func over a pattern of the caller's own
py::object attn_varlen(const py::handle &hq, const py::handle &hk, const py::handle &hv, const py::handle &hcq, const py::handle &hck, int64_t max_q,
                       int64_t max_k, const py::handle &hco, const py::handle &hcn, const py::handle &hind, int64_t lg_m, int64_t lg_n,
                       std::optional<double> softmax_scale, bool causal, bool deterministic) {
  if (!eager()) return none();
  for (const py::handle &h : {hq, hk, hv, hcq, hck, hco, hcn, hind})
    if (!plain(h)) return none();
  const Tensor &q = THPVariable_Unpack(hq.ptr()), &k = THPVariable_Unpack(hk.ptr()), &v = THPVariable_Unpack(hv.ptr());
  const Tensor &cu_q = THPVariable_Unpack(hcq.ptr()), &cu_k = THPVariable_Unpack(hck.ptr());
  Pattern p;
  p.col_offsets = THPVariable_Unpack(hco.ptr()), p.col_nnz = THPVariable_Unpack(hcn.ptr()), p.indices = THPVariable_Unpack(hind.ptr());
  Shape s;
  if (!common_form(s, q, k, cu_q, cu_k, max_q, max_k, lg_n, causal) || !is_rows(v, q.scalar_type(), q.device()) || v.sizes() != k.sizes()) return none();
  if (lg_n % 64 != 0 || lg_m < 128 || lg_m > 1024 || lg_m % 64 != 0) return none();
  for (const Tensor &t : {p.col_offsets, p.col_nnz, p.indices})
    if (t.device() != q.device() || !t.is_contiguous()) return none();
  if (p.col_offsets.scalar_type() != at::kLong || p.col_nnz.scalar_type() != at::kInt || p.indices.scalar_type() != at::kInt || p.col_offsets.dim() != 3 ||
      p.col_offsets.sizes() != p.col_nnz.sizes() || p.col_offsets.size(0) != s.batch || p.col_offsets.size(1) != s.heads || p.col_offsets.size(2) < 1)
    return none();
  s.max_cols = p.col_offsets.size(2);
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  const double scale = softmax_scale ? *softmax_scale : std::pow(static_cast<double>(s.dim), -0.5);
  const int kb = fmoba_attn_fwd_key_block(lg_n);
  // The largest number of visits of a row takes a pass over the lists and a read-back (12037 tokens, 16 heads of 96, 8 of 64-key
  // chunks, forward and backward: a fifth of the call).  It is left out where it cannot change anything: the rules of both forms
  // turn to row blocks and dS tiles as rows get denser, so if the mean (at most list entries per row and head) says so, the
  // maximum does too; and these forms need no bound.  List storage that is larger than the lists raises the mean: dS tiles
  // are sized by the storage, hence the limit on them.
  const int64_t rows = s.total_q * s.heads, mean = std::max<int64_t>(1, (p.indices.numel() + rows - 1) / rows);
  int64_t visits = std::min<int64_t>(mean, s.max_cols) * (lg_n / kb);
  fmoba_attn_fwd_args a = forward_args(s, q, k, v, cu_q, cu_k, visits, scale, nullptr);
  a.col_offsets = p.col_offsets.data_ptr<int64_t>(), a.col_nnz = p.col_nnz.data_ptr<int32_t>(), a.row_indices = p.indices.data_ptr<int32_t>();
  const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
  bool count = !fmoba_attn_fwd_uses_row_blocks(&a);
  if (grad) {
    fmoba_attn_bwd_args b{};
    backward_sizes(b, s, visits * (kb / 64));
    b.num_row_indices = p.indices.numel();
    count = count || fmoba_attn_bwd_uses_partials(&b) || (!capturing && fmoba_attn_bwd_workspace_bytes(&b) > kUncountedBytes);
  }
  // (nothing can be read back while a graph is captured)
  if (count && capturing) return none();
  Tensor out;
  {
    py::gil_scoped_release nogil;
    Result r;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const c10::DeviceGuard guard(q.device());
      check_device(q.device().index());
      s.stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
      if (count) a.max_visits_per_row = visits = count_visits(a, q, s.stream);
      r = forward(s, a, q, p);
    }
    out = grad ? Attention::apply(q, k, v, cu_q, cu_k, p, r, max_q, max_k, lg_n, causal, scale, visits * (kb / 64), deterministic) : r.out;
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

py::tuple last_forward() { return py::make_tuple(t_visits, t_row_blocks); }
int take_last_backward() { return std::exchange(t_partials, -1); }

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  g_parameter_class = py::object(py::module_::import("torch.nn").attr("Parameter")).release().ptr();
  m.def("moba_varlen", &moba_varlen);
  m.def("topk_varlen", &topk_varlen);
  m.def("attn_varlen", &attn_varlen);
  m.def("last_forward", &last_forward);
  m.def("take_last_backward", &take_last_backward);
}
