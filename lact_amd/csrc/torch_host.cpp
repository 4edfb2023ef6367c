// PyTorch side of the operation's calls: checks and converts the tensors, allocates outputs and buffers with torch's
// allocator, enqueues liblact_hip.so on torch's current stream and carries the autograd boundary.  Native because a small
// call (one view rendered, one short sequence) is bound by this code: the same steps in Python cost 65 us of host time per
// forward call and made the GPU wait.  All arithmetic stays behind the C ABI (include/lact_hip.h).
#include <torch/extension.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <memory>
#include <optional>
#include <string>
#include <utility>
#include <vector>

#include "../../include/lact_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A test-time-training schedule (ops.Program) in the C ABI's terms.
struct Schedule : torch::CustomClassHolder {
  std::vector<lact_step_t> steps;
  std::vector<float> coeffs;
  lact_desc_t flags{};          // everything of a descriptor that does not depend on the tensors
  int64_t out_len = 0;
  bool has_update = false, return_state = true, covers = false;

  Schedule(const std::vector<std::vector<int>>& steps_, int64_t out_len_, const std::optional<std::vector<float>>& coeffs_, bool prenorm,
           bool weight_norm, bool detach_norms, bool muon_replaces_weight, int ns_mode, bool muon_stacked, bool renorm_eps_in_sqrt,
           bool return_state_)
      : out_len(out_len_), return_state(return_state_) {
    std::vector<std::pair<int, int>> rows;
    for (const auto& s : steps_) {
      steps.push_back(lact_step_t{s.at(0), s.at(1), s.at(2), s.at(3)});
      if (s[0] == LACT_UPDATE) has_update = true;
      else rows.emplace_back(s[3], s[3] + s[2] - s[1]);
    }
    if (coeffs_) coeffs = *coeffs_;
    flags.n_steps = (int)steps.size();
    flags.out_len = (int)out_len;
    flags.ns_steps = coeffs_ ? (int)coeffs.size() / 3 : -1;
    flags.prenorm = prenorm; flags.weight_norm = weight_norm; flags.detach_norms = detach_norms;
    flags.muon_replaces_weight = muon_replaces_weight; flags.ns_mode = ns_mode;
    flags.muon_stacked = muon_stacked; flags.renorm_eps_in_sqrt = renorm_eps_in_sqrt;
    // do the apply steps write every output row?
    std::sort(rows.begin(), rows.end());
    int pos = 0;
    covers = true;
    for (auto& r : rows) {
      if (r.first > pos) covers = false;
      pos = std::max(pos, r.second);
    }
    covers = covers && pos >= out_len;
  }
};

void check(int rc) {
  if (rc != 0) throw std::runtime_error(std::string("liblact_hip: ") + lact_last_error());
}

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }

// [b, L, d] whose rows the kernels can read with 16-byte vectors.  A clone where they cannot: contiguous() hands back what merely
// starts off a 16-byte boundary or has odd strides in dimensions of size 1.
Tensor rows_view(Tensor t, at::ScalarType dtype) {
  if (t.scalar_type() != dtype) t = t.to(dtype);
  const int64_t align = 16 / t.element_size();
  const bool ok = t.dim() == 3 && t.stride(2) == 1 && t.stride(1) % align == 0 && t.stride(0) % align == 0 && t.stride(1) >= t.size(2) &&
                  t.stride(1) < (1 << 23) && aligned16(t);   // (rows further apart are refused by the library)
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

Tensor plain_f32(const Tensor& t) {
  const Tensor c = t.scalar_type() == at::kFloat ? t.contiguous() : t.to(at::kFloat).contiguous();
  return aligned16(c) ? c : c.clone();
}

Tensor per_token(const Tensor& t, int64_t b, int64_t L, const char* name) {
  if (t.numel() != b * L) {
    std::string s = "(";
    for (auto v : t.sizes()) s += std::to_string(v) + ", ";
    throw std::invalid_argument(std::string(name) + " must hold one value per head and token ([b, l, 1]); got " + s + ")");
  }
  return plain_f32(t.reshape({b, L}));
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
template <typename T = float>
T* fptr(const Tensor& t) { return static_cast<T*>(ptr(t)); }

lact_desc_t describe(const Schedule& sc, int64_t b, int64_t d, int64_t dh, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out) {
  lact_desc_t D = sc.flags;
  D.b = (int)b; D.d = (int)d; D.dh = (int)dh;
  D.q_len = (int)q.size(1); D.kv_len = k.defined() ? (int)k.size(1) : 0;
  D.act_dtype = q.scalar_type() == at::kBFloat16 ? LACT_BF16 : LACT_F32;
  D.steps = sc.steps.data();
  D.ns_coeffs = sc.coeffs.empty() ? nullptr : sc.coeffs.data();
  D.q_bs = q.stride(0); D.q_ld = (int)q.stride(1);
  if (k.defined()) {
    D.k_bs = k.stride(0); D.k_ld = (int)k.stride(1); D.v_bs = v.stride(0); D.v_ld = (int)v.stride(1);
  } else {
    D.k_ld = D.v_ld = (int)d;
  }
  D.o_bs = D.do_bs = out.stride(0); D.o_ld = D.do_ld = (int)out.stride(1);
  return D;
}

struct Operands {      // what a forward call hands to its backward
  Tensor q, k, v, lr0, lr1, lr2, momentum, saved;
  int64_t b = 0, nw = 0, d = 0, dh = 0;
};

// Returns the output, the three final weights (when the schedule returns its state) and the three momentum states (when it
// does and there is momentum).
std::vector<Tensor> forward(const Schedule& sc, const Tensor& w0, const Tensor& w1, const Tensor& w2, const Tensor& q, const OptTensor& k,
                            const OptTensor& v, const OptTensor& lr0, const OptTensor& lr1, const OptTensor& lr2, const OptTensor& momentum,
                            const std::vector<Tensor>& m_state, bool needs_backward, bool shared, Operands* keep) {
  if (!q.is_cuda()) throw std::runtime_error("lact_amd runs on an MI355X only: tensors must be on a HIP device (no CPU path)");
  const c10::hip::HIPGuard guard(q.device().index());
  const int64_t nw = w0.size(0), dh = w0.size(1), d = w0.size(2), b = shared && q.dim() > 0 ? q.size(0) : nw;
  if (w1.sizes() != at::IntArrayRef({nw, d, dh}) || w2.sizes() != at::IntArrayRef({nw, dh, d}))
    throw std::invalid_argument("expected w0, w2: [b, dh, d] and w1: [b, d, dh] with equal key and value dims");
  if (shared && (nw < 1 || b % nw || sc.return_state || !m_state.empty()))
    throw std::invalid_argument("shared weights: their number must divide the batch, and no state is carried in or out");
  // the kernels take raw pointers: a tensor elsewhere, or too small for the steps, has to be refused here
  auto same_device = [&](const Tensor& t) { return t.device() == q.device(); };
  auto here = [&](const OptTensor& t) { return !t || same_device(*t); };
  if (!same_device(w0) || !same_device(w1) || !same_device(w2) || !here(k) || !here(v) || !here(lr0) || !here(lr1) || !here(lr2) || !here(momentum) ||
      !std::all_of(m_state.begin(), m_state.end(), same_device))
    throw std::runtime_error("expected all tensors to be on the same device as q");
  auto is_rows = [&](const Tensor& t) { return t.dim() == 3 && t.size(0) == b && t.size(2) == d; };
  if (!is_rows(q) || (sc.has_update && k && v && (!is_rows(*k) || !is_rows(*v) || v->size(1) < k->size(1))))
    throw std::invalid_argument("expected q, k, v: [b, l, d] with the batch and feature size of the weights, and a row of v for every row of k");
  auto act = (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) ? at::kBFloat16 : at::kFloat;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) act = at::kBFloat16;
  Operands o;
  o.b = b; o.nw = nw; o.d = d; o.dh = dh;
  o.q = rows_view(q, act);
  if (sc.has_update) {
    if (!k || !v || !lr0 || !lr1 || !lr2) throw std::invalid_argument("a schedule with an update needs k, v and the three learning rates");
    o.k = rows_view(*k, act);
    o.v = rows_view(*v, act);
    const int64_t L = o.k.size(1);
    o.lr0 = per_token(*lr0, b, L, "lr");
    o.lr1 = per_token(*lr1, b, L, "lr");
    o.lr2 = per_token(*lr2, b, L, "lr");
    if (momentum) o.momentum = per_token(*momentum, b, L, "momentum");
  }
  // weights that are transposed views of contiguous fp32 tensors (the view-synthesis model's layout) are read as they lie
  auto lies_transposed = [](const Tensor& t) {
    return t.scalar_type() == at::kFloat && t.stride(1) == 1 && t.stride(2) == t.size(1) && t.stride(0) == t.size(1) * t.size(2) && t.size(2) > 1 && aligned16(t);
  };
  const bool transposed = lies_transposed(w0) && lies_transposed(w1) && lies_transposed(w2);
  const Tensor w[3] = {transposed ? w0 : plain_f32(w0), transposed ? w1 : plain_f32(w1), transposed ? w2 : plain_f32(w2)};
  const auto act_opt = o.q.options();
  Tensor out = sc.covers ? at::empty({b, sc.out_len, d}, act_opt) : at::zeros({b, sc.out_len, d}, act_opt);
  lact_desc_t D = describe(sc, b, d, dh, o.q, o.k, o.v, out);
  D.use_momentum = o.momentum.defined();
  D.forward_only = !needs_backward;
  D.w_transposed = transposed;
  Tensor m_in[3];
  const bool carried = !m_state.empty() && o.momentum.defined();
  if (carried) {
    if (needs_backward) throw std::runtime_error("a carried momentum state is an inference feature: call under torch.no_grad()");
    for (int i = 0; i < 3; ++i) {
      m_in[i] = plain_f32(m_state.at(i));
      if (m_in[i].sizes() != w[i].sizes()) throw std::invalid_argument("momentum states must have the shapes of w0, w1, w2");
    }
    D.momentum_state_in = 1;
  }
  size_t saved_bytes = 0, scratch_bytes = 0;
  check(lact_query_sizes(&D, &saved_bytes, &scratch_bytes));
  const auto bytes = act_opt.dtype(at::kByte);
  o.saved = at::empty({(int64_t)saved_bytes}, bytes);
  const Tensor scratch = at::empty({(int64_t)scratch_bytes}, bytes);
  std::vector<Tensor> res{out};
  float* w_out[3] = {nullptr, nullptr, nullptr};
  float* m_out[3] = {nullptr, nullptr, nullptr};
  if (sc.return_state) {
    const int sets = o.momentum.defined() ? 2 : 1;
    for (int i = 0; i < 3 * sets; ++i) res.push_back(at::empty(w[i % 3].sizes(), w[i % 3].options()));
    for (int i = 0; i < 3; ++i) w_out[i] = fptr(res[1 + i]);
    if (o.momentum.defined())
      for (int i = 0; i < 3; ++i) m_out[i] = fptr(res[4 + i]);
  }
  const float* m_ptr[3] = {fptr(m_in[0]), fptr(m_in[1]), fptr(m_in[2])};
  if (shared)
    check(lact_forward_shared_weights(&D, (int)nw, fptr(w[0]), fptr(w[1]), fptr(w[2]), ptr(o.q), ptr(o.k), ptr(o.v), fptr(o.lr0), fptr(o.lr1), fptr(o.lr2),
                                      fptr(o.momentum), ptr(out), w_out, m_out, ptr(o.saved), ptr(scratch), c10::hip::getCurrentHIPStream().stream()));
  else check(lact_forward_from_state(&D, fptr(w[0]), fptr(w[1]), fptr(w[2]), ptr(o.q), ptr(o.k), ptr(o.v), fptr(o.lr0), fptr(o.lr1), fptr(o.lr2),
                                fptr(o.momentum), carried ? m_ptr : nullptr, ptr(out), w_out, m_out, ptr(o.saved), ptr(scratch),
                                c10::hip::getCurrentHIPStream().stream()));
  auto out_dtype = (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kFloat) ? q.scalar_type() : act;
  if (v && v->scalar_type() == at::kFloat && act == at::kBFloat16) out_dtype = at::kFloat;   // zeros_like(v) receives the bf16 products
  if (out_dtype != act) res[0] = out.to(out_dtype);
  if (keep) *keep = std::move(o);
  return res;
}

Tensor cast(const Tensor& t, at::ScalarType dtype) { return !t.defined() || t.scalar_type() == dtype ? t : t.to(dtype); }

// Gradients that have no gradient of their own although they depend on the inputs of the function whose backward is running:
// differentiating them is an error on every path to those inputs, not a silent zero.
void refuse_second_derivative(variable_list& grads) {
  const auto node = torch::autograd::get_current_node();
  const auto err = std::make_shared<torch::autograd::Error>("trying to differentiate twice a function that was marked with @once_differentiable",
                                                            node ? torch::autograd::edge_list(node->next_edges()) : torch::autograd::edge_list());
  for (auto& g : grads)
    if (g.defined()) {
      g = g.detach();
      torch::autograd::create_gradient_edge(g, err);
    }
}
std::vector<OptTensor> refuse_second_derivative_py(std::vector<OptTensor> grads) {
  variable_list list;
  for (auto& g : grads) list.push_back(g ? *g : Tensor());
  refuse_second_derivative(list);
  for (size_t i = 0; i < grads.size(); ++i)
    if (grads[i]) grads[i] = list[i];
  return grads;
}

// What the backward of one call needs beside the saved tensors.
struct CallRecord : torch::CustomClassHolder {
  c10::intrusive_ptr<Schedule> sc;
  int64_t b = 0, nw = 0, d = 0, dh = 0;
  at::ScalarType dtype[8];                 // of w0, w1, w2, q, k, v, the rates, momentum
  std::vector<int64_t> lr_shape, m_shape;
};

struct ProgramFn : torch::autograd::Function<ProgramFn> {
  static variable_list forward(AutogradContext* ctx, c10::intrusive_ptr<Schedule> sc, bool shared, const Tensor& w0, const Tensor& w1, const Tensor& w2,
                               const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& lr0, const OptTensor& lr1,
                               const OptTensor& lr2, const OptTensor& momentum) {
    Operands o;
    auto res = ::forward(*sc, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, {}, true, shared, &o);
    auto rec = c10::make_intrusive<CallRecord>();
    rec->sc = sc;
    rec->b = o.b; rec->nw = o.nw; rec->d = o.d; rec->dh = o.dh;
    auto type = [](const OptTensor& t) { return t ? t->scalar_type() : at::kFloat; };
    const at::ScalarType types[8] = {type(w0), type(w1), type(w2), type(q), type(k), type(v), type(lr0), type(momentum)};
    std::copy(types, types + 8, rec->dtype);
    if (lr0) rec->lr_shape = lr0->sizes().vec();
    if (momentum) rec->m_shape = momentum->sizes().vec();
    ctx->save_for_backward({o.q, o.k, o.v, o.lr0, o.lr1, o.lr2, o.momentum, o.saved});
    ctx->saved_data["call"] = c10::IValue::make_capsule(std::move(rec));
    if (res.size() == 7) ctx->mark_non_differentiable({res[4], res[5], res[6]});
    ctx->set_materialize_grads(false);   // unused outputs arrive undefined in backward, not as zero tensors
    return res;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool twice = at::GradMode::is_enabled();
    const at::AutoGradMode off(false);
    auto t = ctx->get_saved_variables();
    const Tensor &q = t[0], &k = t[1], &v = t[2], &momentum = t[6], &saved = t[7];
    const auto capsule = ctx->saved_data["call"].toCapsule();
    const auto& rec = static_cast<const CallRecord&>(*capsule);
    const Schedule& sc = *rec.sc;
    const int64_t b = rec.b, nw = rec.nw, d = rec.d, dh = rec.dh;
    const c10::hip::HIPGuard guard(q.device().index());
    const auto act_opt = q.options(), f32 = act_opt.dtype(at::kFloat);
    Tensor g_out = grads[0].defined() ? rows_view(grads[0], q.scalar_type()) : at::zeros({b, sc.out_len, d}, act_opt);
    Tensor gw[3];
    const float* gwp[3] = {nullptr, nullptr, nullptr};
    for (size_t i = 0; i < 3 && i + 1 < grads.size(); ++i)
      if (grads[i + 1].defined()) {
        gw[i] = plain_f32(grads[i + 1]);
        gwp[i] = fptr(gw[i]);
      }
    lact_desc_t D = describe(sc, b, d, dh, q, k, v, g_out);
    D.use_momentum = momentum.defined();
    size_t saved_bytes = 0, scratch_bytes = 0;
    check(lact_query_sizes(&D, &saved_bytes, &scratch_bytes));
    const Tensor scratch = at::empty({(int64_t)scratch_bytes}, act_opt.dtype(at::kByte));
    // lact_backward writes every element of its outputs (rows no step touches are zeroed by the library)
    const Tensor dw[3] = {at::empty({nw, dh, d}, f32), at::empty({nw, d, dh}, f32), at::empty({nw, dh, d}, f32)};
    const Tensor dq = at::empty({b, q.size(1), d}, act_opt);
    Tensor dk, dv, dlr[3], dm;
    if (sc.has_update) {
      dk = at::empty({b, k.size(1), d}, act_opt);
      dv = at::empty({b, k.size(1), d}, act_opt);
      for (auto& x : dlr) x = at::empty({b, k.size(1)}, f32);
      if (momentum.defined()) dm = at::empty({b, k.size(1)}, f32);
    }
    check(lact_backward_shared_weights(&D, (int)nw, ptr(q), ptr(k), ptr(v), fptr(t[3]), fptr(t[4]), fptr(t[5]), fptr(momentum), ptr(g_out), gwp, ptr(saved),
                        ptr(scratch), fptr(dw[0]), fptr(dw[1]), fptr(dw[2]), ptr(dq), ptr(dk), ptr(dv), fptr(dlr[0]), fptr(dlr[1]), fptr(dlr[2]),
                        fptr(dm), c10::hip::getCurrentHIPStream().stream()));
    auto type = [&](int i) { return rec.dtype[i]; };
    variable_list res{Tensor(), Tensor(), cast(dw[0], type(0)), cast(dw[1], type(1)), cast(dw[2], type(2)), cast(dq, type(3)), cast(dk, type(4)), cast(dv, type(5))};
    for (auto& x : dlr) res.push_back(x.defined() ? cast(x.reshape(rec.lr_shape), type(6)) : x);
    res.push_back(dm.defined() ? cast(dm.reshape(rec.m_shape), type(7)) : dm);
    if (twice) refuse_second_derivative(res);
    return res;
  }
};

bool wants_grad(const OptTensor& t) { return t && t->requires_grad(); }
bool has_tangent(const Tensor& t) { return t._fw_grad(/*level=*/0).defined(); }
bool has_tangent(const OptTensor& t) { return t && has_tangent(*t); }
template <typename... Ts>
bool any_tangent(const Ts&... ts) { return (has_tangent(ts) || ...); }

// (out, w0, w1, w2, m0, m1, m2), None where there is nothing to return
py::tuple run_program(const c10::intrusive_ptr<Schedule>& sc, const Tensor& w0, const Tensor& w1, const Tensor& w2, const Tensor& q,
                      const OptTensor& k, const OptTensor& v, const OptTensor& lr0, const OptTensor& lr1, const OptTensor& lr2,
                      const OptTensor& momentum, const OptTensor& m0, const OptTensor& m1, const OptTensor& m2, bool shared) {
  // forward-mode differentiation knows nothing of a call that passes the autograd function by: the tangents would be dropped
  if (any_tangent(w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, m0, m1, m2)) {
    PyErr_SetString(PyExc_NotImplementedError, "the operation has no forward-mode derivative (jvp)");
    throw py::error_already_set();
  }
  const bool needs_backward = at::GradMode::is_enabled() &&
                              (w0.requires_grad() || w1.requires_grad() || w2.requires_grad() || q.requires_grad() || wants_grad(k) ||
                               wants_grad(v) || wants_grad(lr0) || wants_grad(lr1) || wants_grad(lr2) || wants_grad(momentum));
  std::vector<Tensor> m_state;
  const bool carries = momentum && sc->has_update;      // otherwise no update would continue from it
  if (m0 && m1 && m2) m_state = {*m0, *m1, *m2};
  else if (carries && (m0 || m1 || m2)) throw std::invalid_argument("a carried momentum state is three tensors, one for each of w0, w1, w2");
  if (needs_backward && !m_state.empty() && carries)
    throw std::runtime_error("a carried momentum state is an inference feature: call under torch.no_grad()");
  variable_list res;
  {
    const py::gil_scoped_release nogil;
    if (needs_backward) {
      res = ProgramFn::apply(sc, shared, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum);
    } else {
      const at::AutoGradMode off(false);
      res = forward(*sc, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, m_state, false, shared, nullptr);
    }
  }
  py::tuple out(7);
  for (size_t i = 0; i < 7; ++i) out[i] = i < res.size() ? py::cast(res[i]) : py::none();
  return out;
}

// ---- the layers' functions around the operation -----------------------------------------------------------------------
// lact_amd/layers.py calls these on plain tensors (its Python functions of the same content take what wants to see Python: hooks,
// transforms, modes).  Native because a layer at a few thousand tokens is bound by its host side: 45 launches and a dozen
// autograd functions per training step took 800 us in Python for 650 us of kernels.
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
Tensor dense(const Tensor& t) {
  const Tensor c = t.contiguous();
  return aligned16(c) ? c : c.clone();
}
Tensor dense(const Tensor& t, at::ScalarType dtype) { return dense(cast(t, dtype)); }
// (in front of a device guard, whose own error names neither the tensor's device nor the reason)
void on_gpu(const Tensor& t) {
  if (!t.is_cuda()) throw std::runtime_error("lact_amd runs on an MI355X only: tensors must be on a HIP device (no CPU path), got one on " + t.device().str());
}
int act_code(const Tensor& t) {
  TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat, "unsupported activation dtype ", t.scalar_type(), ": bf16 or fp32");
  return t.scalar_type() == at::kBFloat16 ? LACT_BF16 : LACT_F32;
}
// The kernels take raw pointers: a tensor elsewhere, or of another shape, has to be refused here.
void expect(const Tensor& t, const Tensor& like, at::IntArrayRef shape, const char* name) {
  if (!t.defined()) return;
  if (t.device() != like.device()) throw std::runtime_error(std::string("expected all tensors to be on the same device: ") + name);
  if (t.sizes() != shape) throw std::invalid_argument(std::string(name) + ": expected shape " + c10::str(shape) + ", got " + c10::str(t.sizes()));
}
Tensor value(const OptTensor& t) { return t ? *t : Tensor(); }
int64_t as_int(AutogradContext* ctx, const char* key) { return ctx->saved_data[key].toInt(); }
// end of every backward: what must not be differentiated again says so
variable_list finish(variable_list grads, bool twice) {
  if (twice) refuse_second_derivative(grads);
  return grads;
}

// qkv [B, L, 3*H*hd] -> q, k, v [(B H), L, hd], and with the rescaling parameters [H*hd, 2] the attention's q, k, v [B, L, H*hd]
struct LayerPreFn : torch::autograd::Function<LayerPreFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv_, const OptTensor& scale_, const OptTensor& offset_, int64_t H, int64_t hd, bool l2norm) {
    on_gpu(qkv_);
    const c10::hip::HIPGuard guard(qkv_.device().index());
    const Tensor qkv = dense(qkv_);
    const int act = act_code(qkv);
    const int64_t B = qkv.size(0), L = qkv.size(1);
    expect(qkv, qkv, {B, L, 3 * H * hd}, "qkv");
    variable_list out;
    for (int i = 0; i < 3; ++i) out.push_back(at::empty({B * H, L, hd}, qkv.options()));
    Tensor scale;
    if (scale_) {
      expect(*scale_, qkv, {H * hd, 2}, "qk_scale");
      expect(*offset_, qkv, {H * hd, 2}, "qk_offset");
      scale = plain_f32(*scale_);
      const Tensor offset = plain_f32(*offset_);
      for (int i = 0; i < 3; ++i) out.push_back(at::empty({B, L, H * hd}, qkv.options()));
      check(lact_layer_pre_attn_forward(act, (int)B, (int)L, (int)H, (int)hd, l2norm, scale_->scalar_type() == qkv.scalar_type(), ptr(qkv), fptr(scale),
                                        fptr(offset), ptr(out[0]), ptr(out[1]), ptr(out[2]), ptr(out[3]), ptr(out[4]), ptr(out[5]), stream()));
      ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)scale_->scalar_type(), (int64_t)offset_->scalar_type()};
    } else {
      check(lact_layer_pre_forward(act, (int)B, (int)L, (int)H, (int)hd, l2norm, ptr(qkv), ptr(out[0]), ptr(out[1]), ptr(out[2]), stream()));
    }
    ctx->save_for_backward({qkv, scale});
    ctx->saved_data["H"] = H; ctx->saved_data["hd"] = hd; ctx->saved_data["l2"] = (int64_t)l2norm;
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool twice = at::GradMode::is_enabled();
    const at::AutoGradMode off(false);
    const auto t = ctx->get_saved_variables();
    const Tensor &qkv = t[0], &scale = t[1];
    const c10::hip::HIPGuard guard(qkv.device().index());
    const int64_t B = qkv.size(0), L = qkv.size(1), H = as_int(ctx, "H"), hd = as_int(ctx, "hd"), l2 = as_int(ctx, "l2");
    for (size_t i = 0; i < grads.size(); ++i)
      grads[i] = grads[i].defined() ? dense(grads[i], qkv.scalar_type())
                                    : i < 3 ? at::zeros({B * H, L, hd}, qkv.options()) : at::zeros({B, L, H * hd}, qkv.options());
    const Tensor dqkv = at::empty_like(qkv);
    variable_list res{dqkv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    if (!scale.defined()) {
      check(lact_layer_pre_backward(act_code(qkv), (int)B, (int)L, (int)H, (int)hd, (int)l2, ptr(qkv), ptr(grads[0]), ptr(grads[1]), ptr(grads[2]), ptr(dqkv), stream()));
    } else {
      const Tensor ds = at::empty_like(scale), doff = at::empty_like(scale);
      const Tensor part = at::empty({lact_layer_pre_attn_part_rows((int)B, (int)L, (int)H) * 4 * H * hd}, scale.options());
      check(lact_layer_pre_attn_backward(act_code(qkv), (int)B, (int)L, (int)H, (int)hd, (int)l2, ptr(qkv), fptr(scale), ptr(grads[0]), ptr(grads[1]), ptr(grads[2]),
                                         ptr(grads[3]), ptr(grads[4]), ptr(grads[5]), ptr(dqkv), fptr(part), fptr(ds), fptr(doff), stream()));
      const auto types = ctx->saved_data["types"].toIntVector();
      res[1] = cast(ds, (at::ScalarType)types[0]);
      res[2] = cast(doff, (at::ScalarType)types[1]);
    }
    return finish(res, twice);
  }
};

// lr_raw [B, L, 3*H], momentum_raw [B, L, H] or none -> lr0, lr1, lr2 (, momentum) [(B H), L, 1] fp32
struct LayerLrFn : torch::autograd::Function<LayerLrFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& lr_, const OptTensor& mom_, int64_t H, double base, bool rates_major) {
    on_gpu(lr_);
    const c10::hip::HIPGuard guard(lr_.device().index());
    const Tensor lr = plain_f32(lr_), mom = mom_ ? plain_f32(*mom_) : Tensor();
    const int64_t B = lr.size(0), L = lr.size(1);
    expect(lr, lr, {B, L, 3 * H}, "lr_raw");
    expect(mom, lr, {B, L, H}, "momentum_raw");
    variable_list out;
    for (int i = 0; i < (mom_ ? 4 : 3); ++i) out.push_back(at::empty({B * H, L, 1}, lr.options()));
    check(lact_layer_lr_forward((int)B, (int)L, (int)H, rates_major, (float)base, fptr(lr), fptr(out[0]), fptr(out[1]), fptr(out[2]), fptr(mom),
                                mom_ ? fptr(out[3]) : nullptr, stream()));
    ctx->save_for_backward({lr, mom});
    ctx->saved_data["H"] = H; ctx->saved_data["base"] = base; ctx->saved_data["major"] = (int64_t)rates_major;
    ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)lr_.scalar_type(), (int64_t)(mom_ ? mom_->scalar_type() : at::kFloat)};
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool twice = at::GradMode::is_enabled();
    const at::AutoGradMode off(false);
    const auto t = ctx->get_saved_variables();
    const Tensor &lr = t[0], &mom = t[1];
    const c10::hip::HIPGuard guard(lr.device().index());
    for (auto& g : grads)
      if (g.defined()) g = plain_f32(g);
    if (grads.size() < 4) grads.resize(4);
    const Tensor dlr = at::empty_like(lr), dmom = mom.defined() ? at::empty_like(mom) : Tensor();
    check(lact_layer_lr_backward((int)lr.size(0), (int)lr.size(1), (int)as_int(ctx, "H"), (int)as_int(ctx, "major"), (float)ctx->saved_data["base"].toDouble(),
                                 fptr(lr), fptr(grads[0]), fptr(grads[1]), fptr(grads[2]), fptr(dlr), fptr(mom), fptr(grads[3]), fptr(dmom), stream()));
    const auto types = ctx->saved_data["types"].toIntVector();
    return finish({cast(dlr, (at::ScalarType)types[0]), cast(dmom, (at::ScalarType)types[1]), Tensor(), Tensor(), Tensor()}, twice);
  }
};

// o [(B H), L, hd] -> y [B, L, H*hd]: RMSNorm per head, times silu(gate_raw [B, L, H]), plus add [B, L, H*hd]
struct LayerPostFn : torch::autograd::Function<LayerPostFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& o_, const OptTensor& weight, const OptTensor& gate, int64_t B, int64_t H, bool use_norm, double eps,
                        const OptTensor& add) {
    on_gpu(o_);
    const c10::hip::HIPGuard guard(o_.device().index());
    const Tensor o = dense(o_);
    const int act = act_code(o);
    const int64_t L = o.size(1), hd = o.size(2);
    expect(o, o, {B * H, L, hd}, "o");
    expect(value(weight), o, {hd}, "weight");
    expect(value(gate), o, {B, L, H}, "gate_raw");
    expect(value(add), o, {B, L, H * hd}, "add");
    const Tensor w = weight ? plain_f32(*weight) : Tensor(), g = gate ? dense(*gate, o.scalar_type()) : Tensor();
    const Tensor a = add ? dense(*add, o.scalar_type()) : Tensor(), y = at::empty({B, L, H * hd}, o.options());
    check(lact_layer_post_add_forward(act, (int)B, (int)L, (int)H, (int)hd, use_norm, (float)eps, ptr(o), fptr(w), ptr(g), ptr(a), ptr(y), stream()));
    ctx->save_for_backward({o, w, g});
    ctx->saved_data["B"] = B; ctx->saved_data["H"] = H; ctx->saved_data["norm"] = (int64_t)use_norm; ctx->saved_data["eps"] = eps;
    auto type = [](const OptTensor& t) { return (int64_t)(t ? t->scalar_type() : at::ScalarType::Undefined); };
    ctx->saved_data["types"] = std::vector<int64_t>{type(weight), type(gate), type(add)};
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool twice = at::GradMode::is_enabled();
    const at::AutoGradMode off(false);
    const auto t = ctx->get_saved_variables();
    const Tensor &o = t[0], &w = t[1], &g = t[2];
    const c10::hip::HIPGuard guard(o.device().index());
    const int64_t B = as_int(ctx, "B"), H = as_int(ctx, "H"), L = o.size(1), hd = o.size(2), norm = as_int(ctx, "norm");
    const Tensor dy = dense(grads[0], o.scalar_type()), d_o = at::empty_like(o), dg = g.defined() ? at::empty_like(g) : Tensor();
    const int64_t rows = lact_layer_post_dw_rows((int)B, (int)L, (int)H);
    const Tensor part = norm && w.defined() ? at::empty({rows, hd}, w.options()) : Tensor();
    check(lact_layer_post_backward(act_code(o), (int)B, (int)L, (int)H, (int)hd, (int)norm, (float)ctx->saved_data["eps"].toDouble(), ptr(o), fptr(w), ptr(g),
                                   ptr(dy), ptr(d_o), ptr(dg), fptr(part), stream()));
    Tensor dw;
    if (part.defined()) {
      dw = at::empty_like(w);
      check(lact_layer_sum_rows((int)rows, (int)hd, fptr(part), fptr(dw), stream()));
    }
    const auto types = ctx->saved_data["types"].toIntVector();
    auto as = [&](const Tensor& x, int i) { return x.defined() && (at::ScalarType)types[i] != at::ScalarType::Undefined ? cast(x, (at::ScalarType)types[i]) : Tensor(); };
    return finish({d_o, as(dw, 0), as(dg, 1), Tensor(), Tensor(), Tensor(), Tensor(), as(grads[0], 2)}, twice);
  }
};

// As autocast casts: a weight once in a region, however often the layer is called there.
Tensor autocast_bf16(const Tensor& t) { return at::autocast::cached_cast(at::kBFloat16, t); }

// a b of bf16 matrices in fp32, inside autocast regions too
Tensor mm_f32(const Tensor& a, const Tensor& b) {
  const c10::impl::ExcludeDispatchKeyGuard plain(c10::DispatchKey::AutocastCUDA);
  return at::mm(a.to(at::kFloat), b.to(at::kFloat));
}
// dy^T x in fp32 for bf16 rows dy [t, m], x [t, n]
Tensor weight_grad(const Tensor& dy, const Tensor& x) {
  const int64_t t = x.size(0), m = dy.size(1), n = x.size(1);
  if (t < 64 || t >= (1LL << 31) || m % 8 || n % 8 || std::max(m, n) >= (1 << 23))   // outside the kernel's range
    return mm_f32(dy.t(), x);
  const Tensor dw = at::empty({m, n}, x.options().dtype(at::kFloat));
  const int64_t bytes = (int64_t)lact_weight_grad_workspace_bytes((int)t, (int)m, (int)n);
  const Tensor ws = bytes ? at::empty({bytes}, x.options().dtype(at::kByte)) : Tensor();
  check(lact_weight_grad((int)t, (int)m, (int)n, ptr(dy), (int)m, ptr(x), (int)n, fptr(dw), ptr(ws), stream()));
  return dw;
}
Tensor rows_of(const Tensor& t, at::ScalarType dtype) { return dense(cast(t, dtype).reshape({-1, t.size(-1)})); }
std::vector<int64_t> with_last(at::IntArrayRef sizes, int64_t last) {
  auto s = sizes.vec();
  s.back() = last;
  return s;
}

// x w^T under bf16 autocast for fp32 w, whose gradient is summed, and returned, in fp32; xb, wb: both as autocast casts them.  It can be
// differentiated again, and over batches of gradients, as the module could: the gradient is then made of torch's operations.
struct LinearFn : torch::autograd::Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& xb, const Tensor& weight, const Tensor& wb) {
    on_gpu(xb);
    const c10::hip::HIPGuard guard(xb.device().index());
    ctx->save_for_backward({xb, wb});
    ctx->saved_data["need"] = std::vector<int64_t>{xb.requires_grad(), weight.requires_grad()};
    return at::linear(dense(xb.reshape({-1, xb.size(-1)})), wb).view(with_last(xb.sizes(), wb.size(0)));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const Tensor &xb = t[0], &wb = t[1];
    const c10::hip::HIPGuard guard(xb.device().index());
    const auto need = ctx->saved_data["need"].toIntVector();
    Tensor dx, dw;
    if (at::GradMode::is_enabled() || grads[0].key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched}))) {
      const Tensor g = grads[0].reshape({-1, wb.size(0)});
      if (need[0]) dx = at::mm(g, wb).view(xb.sizes());
      if (need[1]) dw = mm_f32(g.t(), xb.reshape({-1, xb.size(-1)}));
      return {dx, dw, Tensor()};
    }
    const Tensor g = rows_of(grads[0], at::kBFloat16);
    if (need[0]) dx = at::mm(g, wb).view(xb.sizes());
    if (need[1]) dw = weight_grad(g, rows_of(xb, at::kBFloat16));
    return {dx, dw, Tensor()};
  }
};

// The maps of a layer's input x [B, L, dim] fp32 under bf16 autocast: to_qkv in bf16, the rates x lr_w^T + lr_b in fp32, the bf16
// maps of the momentum (as fp32 values) and of the gate.  to_qkv and the rates are library products; the other maps, and what
// their and the rates' backward is, csrc/layer_kernels.h.  wb: autocast_bf16(qkv_w)
struct LayerInFn : torch::autograd::Function<LayerInFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_, const Tensor& qkv_w, const Tensor& wb, const Tensor& lr_w, const OptTensor& lr_b, const OptTensor& mom_w,
                               const OptTensor& mom_b, const OptTensor& gate_w, const OptTensor& gate_b) {
    on_gpu(x_);
    const c10::hip::HIPGuard guard(x_.device().index());
    const int64_t B = x_.size(0), L = x_.size(1), dim = x_.size(2), n = B * L;
    const Tensor x = rows_of(x_, at::kFloat);
    const Tensor lw = plain_f32(lr_w), mw = mom_w ? plain_f32(*mom_w) : Tensor(), gw = gate_w ? plain_f32(*gate_w) : Tensor();
    const Tensor mb = mom_b ? plain_f32(*mom_b) : Tensor(), gb = gate_b ? plain_f32(*gate_b) : Tensor();
    const int64_t nm = mw.defined() ? mw.size(0) : 0, ng = gw.defined() ? gw.size(0) : 0;
    Tensor lr, mom, gate, xb;
    {
      const c10::impl::ExcludeDispatchKeyGuard plain(c10::DispatchKey::AutocastCUDA);   // the reference keeps the rates out of autocast
      lr = at::linear(x, lw, lr_b ? OptTensor(plain_f32(*lr_b)) : OptTensor());
    }
    if (nm) mom = at::empty({B, L, nm}, x.options());
    if (ng) gate = at::empty({B, L, ng}, wb.options());
    if (nm + ng == 0) {
      xb = x.to(at::kBFloat16);
    } else {
      xb = at::empty({n, dim}, wb.options());
      check(lact_layer_in_forward(n, (int)dim, fptr(x), fptr(mw), fptr(mb), (int)nm, fptr(gw), fptr(gb), (int)ng, ptr(xb), fptr(mom), ptr(gate), stream()));
    }
    ctx->save_for_backward({x, xb, wb, lw, mw, gw});
    auto need = [](const OptTensor& t) { return (int64_t)(t && t->requires_grad()); };
    ctx->saved_data["need"] = std::vector<int64_t>{x_.requires_grad(), qkv_w.requires_grad(), need(lr_w), need(lr_b), need(mom_w), need(mom_b), need(gate_w), need(gate_b)};
    ctx->saved_data["B"] = B; ctx->saved_data["L"] = L;
    ctx->set_materialize_grads(false);
    variable_list out{at::linear(xb, wb).view({B, L, wb.size(0)}), lr.view({B, L, lw.size(0)})};
    if (nm) out.push_back(mom);
    if (ng) out.push_back(gate);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool twice = at::GradMode::is_enabled();
    const at::AutoGradMode off(false);
    const auto t = ctx->get_saved_variables();
    const Tensor &x = t[0], &xb = t[1], &wb = t[2], &lw = t[3], &mw = t[4], &gw = t[5];
    const c10::hip::HIPGuard guard(x.device().index());
    const auto need = ctx->saved_data["need"].toIntVector();
    const int64_t n = x.size(0), dim = x.size(1), counts[3] = {lw.size(0), mw.defined() ? mw.size(0) : 0, gw.defined() ? gw.size(0) : 0};
    Tensor g, dlr, dmom, dgate;
    if (grads[0].defined()) g = rows_of(grads[0], at::kBFloat16);
    if (grads[1].defined()) dlr = plain_f32(grads[1]);
    if (counts[1] && grads[2].defined()) dmom = plain_f32(grads[2]);
    if (counts[2] && grads.back().defined()) dgate = dense(grads.back(), at::kBFloat16);
    Tensor dxq, dx, d[6];
    if (need[0]) {
      dxq = g.defined() ? at::mm(g, wb) : at::zeros_like(xb);
      dx = at::empty({as_int(ctx, "B"), as_int(ctx, "L"), dim}, x.options());
    }
    bool any = false;
    for (int i = 0; i < 6; ++i)
      if (need[2 + i]) {
        d[i] = i % 2 == 0 ? at::empty({counts[i / 2], dim}, x.options()) : at::empty({counts[i / 2]}, x.options());
        any = true;
      }
    const Tensor ws = any ? at::empty({(int64_t)lact_layer_in_backward_workspace_bytes(n, (int)dim, (int)counts[0], (int)counts[1], (int)counts[2])}, x.options().dtype(at::kByte)) : Tensor();
    check(lact_layer_in_backward(n, (int)dim, fptr(x), fptr(lw), (int)counts[0], fptr(mw), (int)counts[1], fptr(gw), (int)counts[2], fptr(dlr), fptr(dmom), ptr(dgate),
                                 ptr(dxq), fptr(dx), fptr(d[0]), fptr(d[1]), fptr(d[2]), fptr(d[3]), fptr(d[4]), fptr(d[5]), ptr(ws), stream()));
    Tensor dw;
    if (need[1]) dw = g.defined() ? weight_grad(g, xb) : at::zeros(wb.sizes(), x.options());
    return finish({dx, dw, Tensor(), d[0], d[1], d[2], d[3], d[4], d[5]}, twice);
  }
};

template <class F, class... Args>
auto apply_released(Args&&... args) {
  const py::gil_scoped_release nogil;
  return F::apply(std::forward<Args>(args)...);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::class_<Schedule, c10::intrusive_ptr<Schedule>>(m, "Schedule")
      .def(py::init<const std::vector<std::vector<int>>&, int64_t, const std::optional<std::vector<float>>&, bool, bool, bool, bool, int, bool,
                    bool, bool>());
  m.def("run_program", &run_program);
  m.def("refuse_second_derivative", &refuse_second_derivative_py);
  m.def("layer_pre", [](const Tensor& qkv, int64_t H, int64_t hd, bool l2norm) { return apply_released<LayerPreFn>(qkv, OptTensor(), OptTensor(), H, hd, l2norm); });
  m.def("layer_pre_attn", [](const Tensor& qkv, const OptTensor& scale, const OptTensor& offset, int64_t H, int64_t hd, bool l2norm) {
    return apply_released<LayerPreFn>(qkv, scale, offset, H, hd, l2norm);
  });
  m.def("layer_lr", [](const Tensor& lr, const OptTensor& mom, int64_t H, double base, bool rates_major) { return apply_released<LayerLrFn>(lr, mom, H, base, rates_major); });
  m.def("layer_post", [](const Tensor& o, const OptTensor& weight, const OptTensor& gate, int64_t B, int64_t H, bool use_norm, double eps, const OptTensor& add) {
    return apply_released<LayerPostFn>(o, weight, gate, B, H, use_norm, eps, add);
  });
  m.def("linear", [](const Tensor& x, const Tensor& weight) { return apply_released<LinearFn>(autocast_bf16(x), weight, autocast_bf16(weight)); });
  m.def("layer_in", [](const Tensor& x, const Tensor& qkv_w, const Tensor& lr_w, const OptTensor& lr_b, const OptTensor& mom_w, const OptTensor& mom_b,
                       const OptTensor& gate_w, const OptTensor& gate_b) { return apply_released<LayerInFn>(x, qkv_w, autocast_bf16(qkv_w), lr_w, lr_b, mom_w, mom_b, gate_w, gate_b); });
}
