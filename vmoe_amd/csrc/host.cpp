// Host side of the layers: the same calls of the C ABI that vmoe_amd/kernels.py makes through
// ctypes, as functions on torch tensors that allocate their results and fill the parameter blocks
// natively.
//
// Why.  A small call is as long as its host work: the sparse layer on one image spends 60 us in
// kernels, and its twenty allocations, forty pointer checks and seven parameter blocks cost 150 us
// of Python (3 us for torch.cuda.current_stream alone, five times a layer).  Here an entry point
// costs its allocations (0.7 us each) and its launch.
//
// Every function takes the raw stream first and raises vmoe_amd._hip.VmoeError on an error code, a
// tensor that is not on the GPU or one that is not contiguous, and ValueError on a tensor with
// another number of axes than its wrapper names or fewer values than the call would read or write
// (TypeError on rows of another type): the C ABI sees addresses and sizes only.  Nothing is kept between calls.
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include <optional>
#include <string>
#include <tuple>

#include "vmoe_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

PyObject* vmoe_error = nullptr;      // vmoe_amd._hip.VmoeError

// (thrown without the interpreter's lock; set_error runs with it)
struct VmoeFailure : py::builtin_exception {
  using builtin_exception::builtin_exception;
  void set_error() const override { PyErr_SetString(vmoe_error != nullptr ? vmoe_error : PyExc_RuntimeError, what()); }
};
struct ZeroDivision : py::builtin_exception {
  using builtin_exception::builtin_exception;
  void set_error() const override { PyErr_SetString(PyExc_ZeroDivisionError, what()); }
};

[[noreturn]] void raise_error(const std::string& text) { throw VmoeFailure(text); }

void check(int code, const char* what) {
  if (code != VMOE_OK)
    raise_error(std::string(what) + " failed: " + vmoe_error_string(code) + " (code " + std::to_string(code) + ")");
}

void* ptr(const Tensor& t) {
  if (!t.is_cuda()) raise_error("tensor is not on a ROCm device; there is no CPU fallback");
  if (!t.is_contiguous()) raise_error("tensor must be contiguous");
  return t.data_ptr();
}
void* ptr(const OptTensor& t) { return t.has_value() ? ptr(*t) : nullptr; }
template <typename T> T* ptr_as(const Tensor& t) { return static_cast<T*>(ptr(t)); }
template <typename T> T* ptr_as(const OptTensor& t) { return static_cast<T*>(ptr(t)); }

std::string shape_of(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + ")";
}
void need_axes(const Tensor& t, int64_t axes, const char* name) {
  if (t.dim() != axes)
    throw py::value_error(std::string(name) + " has shape " + shape_of(t) + ", expected " + std::to_string(axes) +
                          " axes");
}
void need_values(const Tensor& t, int64_t least, const char* name) {
  if (t.numel() < least)
    throw py::value_error(std::string(name) + " has shape " + shape_of(t) + ", expected " + std::to_string(least) + " values");
}
void need_values(const OptTensor& t, int64_t least, const char* name) {
  if (t.has_value()) need_values(*t, least, name);
}
// Two operands that a kernel reads as one type.
void need_type_of(const Tensor& t, const Tensor& like, const char* name, const char* like_name) {
  if (t.scalar_type() != like.scalar_type())
    throw py::type_error(std::string(name) + " is " + at::toString(t.scalar_type()) + ", " + like_name + " " +
                         at::toString(like.scalar_type()));
}
// Stacked weights (at least E, rows, cols).
void need_stack(const OptTensor& t, int64_t E, int64_t rows, int64_t cols, const char* name) {
  if (t.has_value() && (t->dim() != 3 || t->size(0) < E || t->size(1) != rows || t->size(2) != cols))
    throw py::value_error(std::string(name) + " has shape " + shape_of(*t) + ", expected (" + std::to_string(E) + ", " +
                          std::to_string(rows) + ", " + std::to_string(cols) + ")");
}

vmoe_stream_t stream_of(int64_t raw) { return reinterpret_cast<vmoe_stream_t>(raw); }

int dtype_code(at::ScalarType t) {
  if (t == at::kFloat) return VMOE_F32;
  if (t == at::kBFloat16) return VMOE_BF16;
  throw py::type_error("Unsupported dtype; the kernels cover float32 and bfloat16.");
}
int dtype_code(const Tensor& t) { return dtype_code(t.scalar_type()); }

Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const Tensor& like) {
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}
Tensor i32(at::IntArrayRef sizes, const Tensor& like) { return empty(sizes, at::kInt, like); }
Tensor f32(at::IntArrayRef sizes, const Tensor& like) { return empty(sizes, at::kFloat, like); }

Tensor as_f32(const Tensor& t) {     // .to(float32).contiguous() of the wrappers
  return t.scalar_type() == at::kFloat && t.is_contiguous() ? t : t.to(at::kFloat).contiguous();
}

Tensor cast(int64_t stream, const Tensor& x_, at::ScalarType type) {
  if (x_.scalar_type() == type) return x_;
  const Tensor x = x_.contiguous();
  Tensor out = empty(x.sizes(), type, x);
  if (x.numel() > 0) {
    VmoeCastParams p{ptr(x), ptr(out), (size_t)x.numel(), dtype_code(x), dtype_code(type)};
    check(vmoe_cast(&p, stream_of(stream)), "vmoe_cast");
  }
  return out;
}

std::tuple<OptTensor, Tensor, Tensor, OptTensor> gate_topk(
    int64_t stream, const Tensor& x_, const Tensor& w_, int64_t k, const OptTensor& bias_, bool want_gates,
    bool want_logits) {
  need_axes(x_, 3, "x");
  need_axes(w_, 2, "w");
  const Tensor x = x_.contiguous(), w = w_.to(x_.scalar_type()).contiguous();
  const int64_t G = x.size(0), S = x.size(1), D = x.size(2), E = w.size(1);
  need_values(w, D * E, "w");
  need_values(bias_, E, "logit_bias");
  OptTensor bias = bias_;
  if (bias.has_value()) bias = as_f32(*bias);
  OptTensor gates, logits;
  if (want_gates) gates = empty({G, S, E}, x.scalar_type(), x);
  if (want_logits) logits = f32({G, S, E}, x);
  Tensor val = f32({G, S, k}, x), idx = i32({G, S, k}, x);
  VmoeGateTopkParams p{};
  p.x = ptr(x); p.w = ptr(w); p.logit_bias = ptr_as<float>(bias); p.gates = ptr(gates);
  p.topk_val = ptr_as<float>(val); p.topk_idx = ptr_as<int32_t>(idx);
  p.num_items = (int32_t)(G * S); p.D = (int32_t)D; p.E = (int32_t)E; p.K = (int32_t)k;
  p.dtype = dtype_code(x); p.logits = ptr_as<float>(logits);
  check(vmoe_gate_topk(&p, stream_of(stream)), "vmoe_gate_topk");
  return {gates, val, idx, logits};
}

// -> indices, token_slot, slot_token, fill and, with gates, the three losses of the router.
std::tuple<Tensor, Tensor, Tensor, Tensor, OptTensor, OptTensor, OptTensor> route_assign(
    int64_t stream, const OptTensor& val_, const Tensor& idx_, int64_t E, int64_t C, bool batch_priority,
    const OptTensor& gates_, double w_gshard, double w_importance) {
  need_axes(idx_, 3, "topk_idx");
  const Tensor idx = idx_.contiguous();
  OptTensor val = val_, gates = gates_;
  if (val.has_value()) val = as_f32(*val);
  const int64_t G = idx.size(0), S = idx.size(1), K = idx.size(2);
  need_values(val, G * S * K, "topk_val");
  Tensor indices = i32({G, S, K, 2}, idx), token_slot = i32({G, S, K}, idx);
  Tensor slot_token = i32({E * G * C}, idx), fill = i32({G, E}, idx);
  VmoeRouteAssignParams p{};
  p.topk_val = ptr_as<float>(val); p.topk_idx = ptr_as<int32_t>(idx); p.indices = ptr_as<int32_t>(indices);
  p.token_slot = ptr_as<int32_t>(token_slot); p.slot_token = ptr_as<int32_t>(slot_token);
  p.fill = ptr_as<int32_t>(fill);
  p.G = (int32_t)G; p.S = (int32_t)S; p.E = (int32_t)E; p.K = (int32_t)K; p.C = (int32_t)C;
  p.batch_priority = batch_priority;
  OptTensor imp, gsh, aux;
  if (!gates.has_value()) {
    check(vmoe_route_assign(&p, stream_of(stream)), "vmoe_route_assign");
  } else {
    gates = gates->contiguous();
    if (gates->dim() != 3 || gates->size(0) != G || gates->size(1) != S || gates->size(2) != E)
      throw py::value_error("gates do not have the shape (G, S, num_experts)");
    imp = f32({G}, idx); gsh = f32({G}, idx); aux = f32({G}, idx);
    VmoeRouterMetricsParams m{};
    m.gates = ptr(gates); m.top1_idx = ptr_as<int32_t>(idx); m.importance_loss = ptr_as<float>(imp);
    m.gshard_loss = ptr_as<float>(gsh); m.auxiliary_loss = ptr_as<float>(aux);
    m.gshard_loss_weight = (float)w_gshard; m.importance_loss_weight = (float)w_importance;
    m.G = (int32_t)G; m.S = (int32_t)S; m.E = (int32_t)E; m.top1_stride = (int32_t)K; m.dtype = dtype_code(*gates);
    check(vmoe_route_assign_metrics(&p, &m, stream_of(stream)), "vmoe_route_assign_metrics");
  }
  return {indices, token_slot, slot_token, fill, imp, gsh, aux};
}

// Experts-choice routing with its monitoring scalars -> indices, token_slot, slot_token, weights,
// fewest / most experts per item, smallest / largest selected gate, shares of items (num, G), rows
// per expert.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> top_items_metrics(
    int64_t stream, const Tensor& gates_, int64_t C) {
  need_axes(gates_, 3, "gates");
  const Tensor gates = gates_.contiguous();
  const int64_t G = gates.size(0), S = gates.size(1), E = gates.size(2);
  int64_t num = 2;
  while (E >> (num - 1)) ++num;
  Tensor indices = i32({G, S, E, 2}, gates), token_slot = i32({G, S, E}, gates);
  Tensor slot_token = i32({E * G * C}, gates), weights = f32({G, S, E}, gates), sel = f32({G, E, 2}, gates);
  Tensor items = i32({2, G}, gates), gate = empty({2, G}, gates.scalar_type(), gates);
  Tensor ratios = f32({num, G}, gates), rows = i32({E}, gates);
  VmoeTopItemsParams p{ptr(gates), ptr_as<int32_t>(indices), ptr_as<int32_t>(token_slot),
                       ptr_as<int32_t>(slot_token), ptr_as<float>(weights), ptr_as<float>(sel), (int32_t)G,
                       (int32_t)S, (int32_t)E, (int32_t)C, dtype_code(gates)};
  check(vmoe_top_items_metrics(&p, ptr_as<int32_t>(items), ptr(gate), ptr_as<float>(ratios),
                               ptr_as<int32_t>(rows), stream_of(stream)), "vmoe_top_items_metrics");
  return {indices, token_slot, slot_token, weights, items, gate, ratios, rows};
}

// The expert MLP; with `fill` and `token_slot` the packed rows are computed here as well.
// -> out, workspace, byte offset of the status words in it (-1: none), token_row,
//    rows_per_expert, row_token, whether the call ran on a plan that the compaction wrote.
std::tuple<Tensor, Tensor, int64_t, OptTensor, OptTensor, OptTensor, bool> expert_mlp(
    int64_t stream, const Tensor& x_, const OptTensor& w0, const OptTensor& b0_, const OptTensor& w1,
    const OptTensor& b1_, const OptTensor& w0t, const OptTensor& w1t, bool tanh_gelu,
    const OptTensor& workspace_, const OptTensor& out_, const OptTensor& rows_per_expert,
    const OptTensor& x_rows, const OptTensor& fill, const OptTensor& token_slot, int64_t capacity,
    bool plan_apart, bool f32_products, bool full_rows) {
  const Tensor x = x_.contiguous();
  // float32 biases of a bfloat16 MLP are rounded by the call (which asks for both in one type)
  auto is_f32 = [&](const OptTensor& t) { return t.has_value() && t->scalar_type() == at::kFloat; };
  const bool f32_biases = x.scalar_type() == at::kBFloat16 && (is_f32(b0_) || is_f32(b1_));
  auto bias = [&](const OptTensor& t) -> OptTensor {
    return f32_biases && t.has_value() ? OptTensor(as_f32(*t)) : t;
  };
  const OptTensor b0 = bias(b0_), b1 = bias(b1_);
  const bool compact = fill.has_value();
  VmoeCompactRowsParams c{};
  OptTensor token_row, rows = rows_per_expert, row_token = x_rows;
  if (compact) {
    need_axes(*fill, 2, "fill");
    need_axes(*token_slot, 3, "token_slot");
    need_values(*token_slot, fill->size(0) * token_slot->size(1) * token_slot->size(2), "token_slot");
    c.G = (int32_t)fill->size(0); c.E = (int32_t)fill->size(1); c.C = (int32_t)capacity;
    c.S = (int32_t)token_slot->size(1); c.K = (int32_t)token_slot->size(2);
    token_row = i32({c.G, c.S, c.K}, *fill);
    rows = i32({c.E}, *fill);
    row_token = i32({c.E, c.G * capacity}, *fill);
    c.fill = ptr_as<int32_t>(fill); c.token_slot = ptr_as<int32_t>(token_slot);
    c.token_row = ptr_as<int32_t>(token_row); c.rows_per_expert = ptr_as<int32_t>(rows);
    c.row_token = ptr_as<int32_t>(row_token);
  }
  VmoeExpertMlpParams p{};
  int64_t E, R, D;
  need_axes(x, row_token.has_value() ? 2 : 3, "x");
  if (row_token.has_value()) {
    need_axes(*row_token, 2, "x_rows");
    E = row_token->size(0); R = row_token->size(1);
    p.num_items = (int32_t)x.size(0); D = x.size(1);
  } else {
    E = x.size(0); R = x.size(1); D = x.size(2);
  }
  p.E = (int32_t)E; p.R = (int32_t)R; p.D = (int32_t)D;
  const OptTensor& first = w0.has_value() ? w0 : w0t;
  if (!first.has_value()) throw py::value_error("neither w0 nor w0t is given");
  need_axes(*first, 3, w0.has_value() ? "w0" : "w0t");
  const int64_t M = first->size(w0.has_value() ? 2 : 1);
  need_stack(w0, E, D, M, "w0");
  need_stack(w0t, E, M, D, "w0t");
  need_stack(w1, E, M, D, "w1");
  need_stack(w1t, E, D, M, "w1t");
  need_values(b0, E * M, "b0");
  need_values(b1, E * D, "b1");
  need_values(rows, E, "rows_per_expert");
  need_values(out_, E * R * D, "out");
  p.M = (int32_t)M;
  Tensor out = out_.has_value() ? *out_ : empty({E, R, D}, x.scalar_type(), x);
  p.x = ptr(x); p.w0 = ptr(w0); p.b0 = ptr(b0); p.w1 = ptr(w1); p.b1 = ptr(b1); p.w0t = ptr(w0t); p.w1t = ptr(w1t);
  p.out = ptr(out); p.dtype = dtype_code(x);
  p.gelu = (tanh_gelu ? VMOE_GELU_TANH : VMOE_GELU_ERF) + (f32_products ? VMOE_MLP_F32_PRODUCTS : 0) +
           (f32_biases ? VMOE_MLP_F32_BIASES : 0) + (full_rows ? VMOE_MLP_FULL_ROWS : 0);
  p.rows_per_expert = ptr_as<int32_t>(rows); p.x_rows = ptr_as<int32_t>(row_token);
  const size_t need = vmoe_expert_mlp_workspace_bytes(&p);
  Tensor workspace = workspace_.has_value() && workspace_->nbytes() >= need
                         ? *workspace_ : empty({(int64_t)need}, at::kByte, x);
  p.workspace = ptr(workspace);
  p.workspace_bytes = workspace.nbytes();
  const int32_t* status = nullptr;
  check(vmoe_expert_mlp_status(&p, &status), "vmoe_expert_mlp_status");
  const int64_t status_at = status == nullptr ? -1 : (const char*)status - (const char*)p.workspace;
  if (compact) {
    int rc = VMOE_E_UNSUPPORTED;
    if (p.dtype == VMOE_BF16 && !plan_apart) rc = vmoe_compact_rows_planned(&c, &p, stream_of(stream));
    if (rc == VMOE_OK) {
      check(vmoe_expert_mlp_planned(&p, stream_of(stream)), "vmoe_expert_mlp_planned");
      return {out, workspace, status_at, token_row, rows, row_token, true};
    }
    if (rc != VMOE_E_UNSUPPORTED) check(rc, "vmoe_compact_rows_planned");
    const Tensor prefix = i32({c.G, c.E}, *fill);
    c.prefix = ptr_as<int32_t>(prefix);
    check(vmoe_compact_rows(&c, stream_of(stream)), "vmoe_compact_rows");
  }
  check(vmoe_expert_mlp(&p, stream_of(stream)), "vmoe_expert_mlp");
  return {out, workspace, status_at, token_row, rows, row_token, false};
}

Tensor dispatch(int64_t stream, const Tensor& x_, const Tensor& token_slot, const OptTensor& slot_token,
                const OptTensor& out_, std::optional<int64_t> slots) {
  need_axes(x_, 2, "x");
  const Tensor x = x_.contiguous();
  const int64_t D = x.size(1);
  if (!slot_token.has_value() && !slots.has_value()) throw py::type_error("dispatch needs slot_token or num_slots");
  const int64_t num_slots = slot_token.has_value() ? slot_token->numel() : *slots;
  if (token_slot.dim() < 1) need_axes(token_slot, 2, "token_slot");
  need_values(token_slot, x.size(0) * token_slot.size(-1), "token_slot");
  need_values(out_, num_slots * D, "out");
  Tensor out = out_.has_value() ? *out_ : empty({num_slots, D}, x.scalar_type(), x);
  VmoeDispatchParams p{ptr(x), ptr_as<int32_t>(token_slot), ptr_as<int32_t>(slot_token), ptr(out),
                       (int32_t)x.size(0), (int32_t)num_slots, (int32_t)token_slot.size(-1), (int32_t)D,
                       dtype_code(x)};
  check(vmoe_dispatch(&p, stream_of(stream)), "vmoe_dispatch");
  return out;
}

Tensor combine(int64_t stream, const Tensor& y_, const Tensor& token_slot, const Tensor& weights_,
               const OptTensor& out_) {
  need_axes(y_, 2, "y");
  need_axes(token_slot, 2, "token_slot");
  const Tensor y = y_.contiguous(), weights = as_f32(weights_);
  const int64_t D = y.size(1), T = token_slot.size(0);
  need_values(weights, token_slot.numel(), "weights");
  need_values(out_, T * D, "out");
  Tensor out = out_.has_value() ? *out_ : empty({T, D}, y.scalar_type(), y);
  VmoeCombineParams p{ptr(y), ptr_as<int32_t>(token_slot), ptr_as<float>(weights), ptr(out), (int32_t)T,
                      (int32_t)y.size(0), (int32_t)token_slot.size(1), (int32_t)D, dtype_code(y)};
  check(vmoe_combine(&p, stream_of(stream)), "vmoe_combine");
  return out;
}

// -> (x, layer_norm(x)): x the residual itself without a branch.
std::tuple<Tensor, OptTensor> add_layer_norm(int64_t stream, const Tensor& residual_, const OptTensor& branch_,
                                             const OptTensor& scale_, const OptTensor& bias_, double eps,
                                             std::optional<at::ScalarType> out_type, bool write_residual) {
  if (residual_.dim() < 1) need_axes(residual_, 1, "residual");
  if (residual_.size(-1) == 0) throw ZeroDivision("residual has an empty last axis");   // (rows are a quotient)
  const Tensor residual = residual_.contiguous();
  OptTensor branch = branch_, scale = scale_, bias = bias_, sum, norm;
  const int64_t D = residual.size(-1);
  if (branch.has_value()) {
    if (branch->sizes() != residual.sizes()) throw py::value_error("branch and residual have different shapes");
    branch = branch->contiguous();
    if (write_residual) sum = at::empty_like(residual);
  }
  need_values(scale, D, "scale");
  need_values(bias, D, "bias");
  if (scale.has_value()) scale = as_f32(*scale);
  if (bias.has_value()) bias = as_f32(*bias);
  if (out_type.has_value()) norm = empty(residual.sizes(), *out_type, residual);
  if (!sum.has_value() && !norm.has_value()) return {residual, norm};
  VmoeAddLayerNormParams p{ptr_as<float>(residual), ptr(branch), ptr_as<float>(scale), ptr_as<float>(bias),
                           ptr_as<float>(sum), ptr(norm), (size_t)(residual.numel() / D), (int32_t)D, (float)eps,
                           branch.has_value() ? dtype_code(*branch) : 0,
                           out_type.has_value() ? dtype_code(*out_type) : 0};
  check(vmoe_add_layer_norm(&p, stream_of(stream)), "vmoe_add_layer_norm");
  return {sum.has_value() ? *sum : residual, norm};
}

Tensor attention(int64_t stream, const Tensor& q, const Tensor& k, const Tensor& v, double scale) {
  need_axes(q, 4, "q");
  need_axes(k, 4, "k");
  need_axes(v, 4, "v");
  const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), hd = q.size(3);
  for (const Tensor* t : {&k, &v})
    if (t->size(0) < B || t->size(1) < k.size(1) || t->size(2) < H)
      throw py::value_error("keys or values of shape " + shape_of(*t) + " for queries of shape " + shape_of(q));
  for (const Tensor* t : {&q, &k, &v}) {
    if (!t->is_cuda()) raise_error("tensor is not on a ROCm device; there is no CPU fallback");
    if (t->stride(3) != 1 || t->stride(2) != hd)
      raise_error("attention operands need contiguous (H, hd) trailing axes");
  }
  Tensor out = empty({B, Sq, H * hd}, q.scalar_type(), q);
  VmoeAttentionParams p{q.data_ptr(), k.data_ptr(), v.data_ptr(), ptr(out), q.stride(0), q.stride(1), k.stride(0),
                        k.stride(1), v.stride(0), v.stride(1), (int32_t)B, (int32_t)H, (int32_t)Sq,
                        (int32_t)k.size(1), (int32_t)hd, (float)scale, dtype_code(q)};
  check(vmoe_attention(&p, stream_of(stream)), "vmoe_attention");
  return out;
}

int w_code(const Tensor& w) {
  switch (w.scalar_type()) {
    case at::kFloat: return VMOE_W_F32;
    case at::kBFloat16: return VMOE_W_BF16;
    case at::kBool: return VMOE_W_BOOL;
    default: break;
  }
  throw py::type_error("Unsupported weight dtype");
}

// Dense dispatch (G, S, E, C) x (G, S, D) -> (E*G*C, D), or combine -> (G, S, D).
// rounded: float32 data, rounded to bfloat16 as they are read.
Tensor einsum(int64_t stream, const Tensor& w_, const Tensor& data_, at::ScalarType out_type, bool is_dispatch,
              bool rounded) {
  need_axes(w_, 4, "w");
  if (data_.dim() < 1) need_axes(data_, is_dispatch ? 3 : 2, "data");
  const Tensor w = w_.contiguous(), data = data_.contiguous();
  const int64_t G = w.size(0), S = w.size(1), E = w.size(2), C = w.size(3), D = data.size(-1);
  need_values(data, (is_dispatch ? G * S : E * G * C) * D, "data");
  Tensor out = is_dispatch ? empty({E * G * C, D}, out_type, data) : empty({G, S, D}, out_type, data);
  VmoeEinsumParams p{ptr(w), ptr(data), ptr(out), (int32_t)G, (int32_t)S, (int32_t)E, (int32_t)C, (int32_t)D,
                     w_code(w), rounded && data.scalar_type() == at::kFloat ? VMOE_EINSUM_F32_AS_BF16 : dtype_code(data),
                     dtype_code(out_type)};
  if (is_dispatch) check(vmoe_einsum_dispatch(&p, stream_of(stream)), "vmoe_einsum_dispatch");
  else check(vmoe_einsum_combine(&p, stream_of(stream)), "vmoe_einsum_combine");
  return out;
}

// -> dispatch weights, combine weights, the (5,) scalars of the weights, the prepared slot
// parameters (`prepared`, if given, is what an earlier call with the same mu, scale and shapes left).
std::tuple<Tensor, Tensor, Tensor, Tensor> soft_route_stats(int64_t stream, const Tensor& x_, const Tensor& mu_,
                                                            double scale, const OptTensor& prepared) {
  need_axes(x_, 3, "x");
  need_axes(mu_, 2, "mu");
  const Tensor x = x_.contiguous(), mu = mu_.to(x_.scalar_type()).contiguous();
  const int64_t G = x.size(0), S = x.size(1), D = x.size(2), N = mu.size(1);
  need_values(mu, D * N, "mu");
  Tensor dw = empty({G, S, N}, x.scalar_type(), x), cw = empty({G, S, N}, x.scalar_type(), x);
  Tensor buf = f32({G * 4 + 8}, x);
  VmoeSoftRouteParams p{};
  p.x = ptr(x); p.mu = ptr(mu); p.scale = (float)scale; p.dispatch_w = ptr(dw); p.combine_w = ptr(cw);
  p.G = (int32_t)G; p.S = (int32_t)S; p.D = (int32_t)D; p.N = (int32_t)N; p.dtype = dtype_code(x);
  Tensor ws = prepared.has_value() ? *prepared
                                   : empty({std::max<int64_t>(16, vmoe_soft_route_workspace_bytes(&p))}, at::kByte, x);
  p.workspace = ptr(ws); p.workspace_bytes = ws.nbytes(); p.workspace_prepared = prepared.has_value();
  VmoeSoftStatsParams st{p.combine_w, p.dispatch_w, ptr_as<float>(buf), ptr_as<float>(buf) + G * 4, p.G, p.S, p.N, p.dtype};
  check(vmoe_soft_route_stats(&p, &st, stream_of(stream)), "vmoe_soft_route_stats");
  return {dw, cw, buf.slice(0, G * 4, G * 4 + 5), ws};
}

// -> dy (data) or dweights (weights) of combine.
Tensor combine_backward_data(int64_t stream, const Tensor& dout_, const Tensor& token_slot, const Tensor& weights_,
                             const OptTensor& slot_token, int64_t num_slots) {
  need_axes(dout_, 2, "dout");
  if (token_slot.dim() < 1) need_axes(token_slot, 2, "token_slot");
  const Tensor dout = dout_.contiguous(), weights = as_f32(weights_);
  need_values(token_slot, dout.size(0) * token_slot.size(-1), "token_slot");
  need_values(weights, dout.size(0) * token_slot.size(-1), "weights");
  need_values(slot_token, num_slots, "slot_token");
  Tensor dy = empty({num_slots, dout.size(1)}, dout.scalar_type(), dout);
  VmoeCombineBackwardParams p{};
  p.dout = ptr(dout); p.token_slot = ptr_as<int32_t>(token_slot); p.weights = ptr_as<float>(weights);
  p.slot_token = ptr_as<int32_t>(slot_token); p.dy = ptr(dy);
  p.num_items = (int32_t)dout.size(0); p.num_slots = (int32_t)num_slots; p.K = (int32_t)token_slot.size(-1);
  p.D = (int32_t)dout.size(1); p.dtype = dtype_code(dout);
  check(vmoe_combine_backward_data(&p, stream_of(stream)), "vmoe_combine_backward_data");
  return dy;
}

Tensor combine_backward_weights(int64_t stream, const Tensor& dout_, const Tensor& y_, const Tensor& token_slot) {
  need_axes(dout_, 2, "dout");
  need_axes(y_, 2, "y");
  if (token_slot.dim() < 1) need_axes(token_slot, 2, "token_slot");
  const Tensor dout = dout_.contiguous(), y = y_.contiguous();
  need_values(token_slot, dout.size(0) * token_slot.size(-1), "token_slot");
  need_values(y, y.size(0) * dout.size(1), "y");
  need_type_of(y, dout, "y", "dout");
  Tensor dw = f32({dout.size(0), token_slot.size(-1)}, dout);
  VmoeCombineBackwardParams p{};
  p.dout = ptr(dout); p.y = ptr(y); p.token_slot = ptr_as<int32_t>(token_slot); p.dweights = ptr_as<float>(dw);
  p.num_items = (int32_t)dout.size(0); p.num_slots = (int32_t)y.size(0); p.K = (int32_t)token_slot.size(-1);
  p.D = (int32_t)dout.size(1); p.dtype = dtype_code(dout);
  check(vmoe_combine_backward_weights(&p, stream_of(stream)), "vmoe_combine_backward_weights");
  return dw;
}

// -> (dy, dweights) of combine.
std::tuple<Tensor, Tensor> combine_backward(int64_t stream, const Tensor& dout_, const Tensor& y_, const Tensor& token_slot,
                                            const Tensor& weights_, const OptTensor& slot_token) {
  need_axes(dout_, 2, "dout");
  need_axes(y_, 2, "y");
  if (token_slot.dim() < 1) need_axes(token_slot, 2, "token_slot");
  const Tensor dout = dout_.contiguous(), y = y_.contiguous(), weights = as_f32(weights_);
  need_values(token_slot, dout.size(0) * token_slot.size(-1), "token_slot");
  need_values(weights, dout.size(0) * token_slot.size(-1), "weights");
  need_values(slot_token, y.size(0), "slot_token");
  need_values(y, y.size(0) * dout.size(1), "y");
  need_type_of(y, dout, "y", "dout");
  Tensor dy = empty({y.size(0), dout.size(1)}, dout.scalar_type(), dout);
  Tensor dw = f32({dout.size(0), token_slot.size(-1)}, dout);
  VmoeCombineBackwardParams p{};
  p.dout = ptr(dout); p.y = ptr(y); p.token_slot = ptr_as<int32_t>(token_slot); p.weights = ptr_as<float>(weights);
  p.slot_token = ptr_as<int32_t>(slot_token); p.dy = ptr(dy); p.dweights = ptr_as<float>(dw);
  p.num_items = (int32_t)dout.size(0); p.num_slots = (int32_t)y.size(0); p.K = (int32_t)token_slot.size(-1);
  p.D = (int32_t)dout.size(1); p.dtype = dtype_code(dout);
  check(vmoe_combine_backward(&p, stream_of(stream)), "vmoe_combine_backward");
  return {dy, dw};
}

// x (..., D) . w + b -> (..., M), rounded once: float32 w (D, M), bfloat16 w transposed (M, D).
Tensor dense(int64_t stream, const Tensor& x_, const Tensor& w_, const OptTensor& b_) {
  if (x_.dim() < 2) need_axes(x_, 2, "x");
  need_axes(w_, 2, "w");
  need_type_of(w_, x_, "w", "x");
  if (b_.has_value()) need_type_of(*b_, x_, "bias", "x");
  const Tensor x = x_.contiguous(), w = w_.contiguous();
  const OptTensor b = b_.has_value() ? OptTensor(b_->contiguous()) : b_;
  const bool f32 = x.scalar_type() == at::kFloat;
  const int64_t D = x.size(-1), M = w.size(f32 ? 1 : 0);
  if (w.size(f32 ? 0 : 1) != D || D == 0)
    throw py::value_error("w has shape " + shape_of(w) + ", x " + shape_of(x));
  if (b.has_value() && b->numel() != M)
    throw py::value_error("bias has shape " + shape_of(*b) + ", expected (" + std::to_string(M) + ",)");
  if (x.numel() / D > INT32_MAX) throw py::value_error("x has shape " + shape_of(x) + ": too many rows");
  auto sizes = x.sizes().vec();
  sizes.back() = M;
  Tensor out = empty(sizes, x.scalar_type(), x);
  if (out.numel() == 0) return out;
  VmoeExpertMlpParams p{};
  p.x = ptr(x); (f32 ? p.w0 : p.w0t) = ptr(w); p.b0 = ptr(b); p.out = ptr(out);
  p.E = 1; p.R = (int32_t)(x.numel() / D); p.D = (int32_t)D; p.M = (int32_t)M; p.dtype = dtype_code(x);
  check(vmoe_dense(&p, stream_of(stream)), "vmoe_dense");
  return out;
}

// -> dx of dispatch.
Tensor dispatch_backward(int64_t stream, const Tensor& dbuf_, const Tensor& token_slot) {
  need_axes(dbuf_, 2, "dbuf");
  need_axes(token_slot, 2, "token_slot");
  const Tensor dbuf = dbuf_.contiguous();
  const int64_t D = dbuf.size(1), T = token_slot.size(0);
  Tensor dx = empty({T, D}, dbuf.scalar_type(), dbuf);
  VmoeCombineParams p{ptr(dbuf), ptr_as<int32_t>(token_slot), nullptr, ptr(dx), (int32_t)T, (int32_t)dbuf.size(0),
                      (int32_t)token_slot.size(1), (int32_t)D, dtype_code(dbuf)};
  check(vmoe_dispatch_backward(&p, stream_of(stream)), "vmoe_dispatch_backward");
  return dx;
}

// dispatch and combine with their gradients, for autograd's own threads: a backward pass through
// Python functions waits for the interpreter in every node (a pass over 128 images of 196 tokens, both
// directions: 160 us of host work for 118 of kernels).  The same nodes as moe.py's _DispatchFn and
// _CombineFn, which stand in wherever something besides autograd looks on.
int64_t current_stream() { return reinterpret_cast<int64_t>(c10::hip::getCurrentHIPStream().stream()); }

struct DispatchFn : torch::autograd::Function<DispatchFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& rows, const Tensor& token_slot,
                        const Tensor& slot_token) {
    ctx->save_for_backward({token_slot});
    return dispatch(current_stream(), rows, token_slot, slot_token, std::nullopt, std::nullopt);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    return {dispatch_backward(current_stream(), grads[0], saved[0]), Tensor(), Tensor()};
  }
};

struct CombineFn : torch::autograd::Function<CombineFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& rows, const Tensor& token_slot,
                        const Tensor& weights, const Tensor& slot_token) {
    ctx->save_for_backward({rows, token_slot, weights, slot_token});
    return combine(current_stream(), rows, token_slot, weights, std::nullopt);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &rows = saved[0], &token_slot = saved[1], &weights = saved[2], &slot_token = saved[3];
    const Tensor grad = grads[0].contiguous();
    Tensor d_rows, d_weights;
    if (ctx->needs_input_grad(0) && ctx->needs_input_grad(2) && grad.scalar_type() == rows.scalar_type()) {
      std::tie(d_rows, d_weights) = combine_backward(current_stream(), grad, rows, token_slot, weights, slot_token);
    } else {
      if (ctx->needs_input_grad(0))
        d_rows = combine_backward_data(current_stream(), grad, token_slot, weights, slot_token, rows.size(0));
      if (ctx->needs_input_grad(2)) d_weights = combine_backward_weights(current_stream(), grad, rows, token_slot);
    }
    if (d_weights.defined()) d_weights = d_weights.to(weights.scalar_type());
    return {d_rows, Tensor(), d_weights, Tensor()};
  }
};

Tensor dispatch_recorded(const Tensor& rows, const Tensor& token_slot, const Tensor& slot_token) {
  return DispatchFn::apply(rows, token_slot, slot_token);
}
Tensor combine_recorded(const Tensor& rows, const Tensor& token_slot, const Tensor& weights, const Tensor& slot_token) {
  return CombineFn::apply(rows, token_slot, weights, slot_token);
}

// -> (token_slot (G, S, K), slot_token (E * G * C,), counters (2,): duplicates, invalid).
std::tuple<Tensor, Tensor, Tensor> indices_to_slots(int64_t stream, const Tensor& indices_, int64_t E, int64_t C) {
  need_axes(indices_, 4, "indices");
  const Tensor indices = indices_.to(at::kInt).contiguous();
  const int64_t G = indices.size(0), S = indices.size(1), K = indices.size(2);
  need_values(indices, 2 * G * S * K, "indices");
  const auto i32 = indices.options();
  Tensor token_slot = at::empty({G, S, K}, i32), slot_token = at::empty({E * G * C}, i32), counters = at::empty({2}, i32);
  int32_t* const counts = ptr_as<int32_t>(counters);
  VmoeIndicesToSlotsParams p{ptr_as<int32_t>(indices), ptr_as<int32_t>(token_slot), ptr_as<int32_t>(slot_token), counts,
                             counts + 1, (int32_t)G, (int32_t)S, (int32_t)E, (int32_t)K, (int32_t)C};
  check(vmoe_indices_to_slots(&p, stream_of(stream)), "vmoe_indices_to_slots");
  return {token_slot, slot_token, counters};
}

}  // namespace

// Calls run without the interpreter's lock, as ctypes makes them (a launch can wait for room in the
// queue, an allocation for the device).
#define VMOE_DEF(name) m.def(#name, torch::wrap_pybind_function_no_gil(&name))

PYBIND11_MODULE(_vmoe_host, m) {
  m.def("set_error", [](py::object e) { vmoe_error = e.release().ptr(); });
  m.def("cast", [](int64_t s, const Tensor& x, py::object t) {
    return torch::wrap_pybind_function_no_gil(&cast)(s, x, torch::python::detail::py_object_to_dtype(std::move(t)));
  });
  VMOE_DEF(gate_topk);
  VMOE_DEF(route_assign);
  VMOE_DEF(top_items_metrics);
  VMOE_DEF(expert_mlp);
  VMOE_DEF(dispatch);
  VMOE_DEF(combine);
  m.def("add_layer_norm", [](int64_t s, const Tensor& r, const OptTensor& b, const OptTensor& sc, const OptTensor& bi,
                             double eps, py::object t, bool w) {
    std::optional<at::ScalarType> type;
    if (!t.is_none()) type = torch::python::detail::py_object_to_dtype(std::move(t));
    return torch::wrap_pybind_function_no_gil(&add_layer_norm)(s, r, b, sc, bi, eps, type, w);
  });
  VMOE_DEF(attention);
  VMOE_DEF(dense);
  m.def("einsum", [](int64_t s, const Tensor& w, const Tensor& d, py::object t, bool dispatch_, bool rounded) {
    return torch::wrap_pybind_function_no_gil(&einsum)(s, w, d, torch::python::detail::py_object_to_dtype(std::move(t)),
                                                       dispatch_, rounded);
  });
  VMOE_DEF(soft_route_stats);
  VMOE_DEF(combine_backward_data);
  VMOE_DEF(combine_backward_weights);
  VMOE_DEF(combine_backward);
  VMOE_DEF(dispatch_backward);
  VMOE_DEF(dispatch_recorded);
  VMOE_DEF(combine_recorded);
  VMOE_DEF(indices_to_slots);
}
