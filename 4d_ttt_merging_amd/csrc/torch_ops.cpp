// The CUDA (HIP) implementations of the torch operators `torch.ops.vgo.*`
// (schemas: ops.py), calling the C ABI of libvgo.so.
//
// Native so that a call costs its launches and little else: with the operators
// implemented in Python (argument boxing in and out of the dispatcher, two
// Python autograd layers, ctypes), a residual row pass took 24 us of host time and
// an attention call 19 us, more than their kernels at small sizes.
//
// Every implementation checks shapes and types, allocates outputs and
// workspaces with torch, and launches on torch's current stream of the
// tensors' device, which is the current device meanwhile (`on_device`); none
// synchronises.  Autograd: outputs of a path operator whose inputs
// require grad have a backward that raises (the path is inference only), those
// of a planner's operator do not require grad, and tangents are dropped.
// No operator has a batching rule (see register_batched).
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/library.h>

#include <array>
#include <memory>
#include <optional>
#include <string>
#include <vector>

#include "../../include/vgo.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// Status of a C call as the exception the reference's call would raise.
void check(int status) {
  if (status == VGO_OK) return;
  const std::string message = vgo_last_error();
  if (status == VGO_EINVAL) TORCH_CHECK_VALUE(false, message);
  TORCH_CHECK(false, message);
}

void require_gpu(std::initializer_list<const Tensor*> tensors) {
  for (const Tensor* t : tensors)
    TORCH_CHECK(t == nullptr || !t->defined() || t->is_cuda(), "vgo kernels run on the GPU only; got a CPU tensor");
}
const Tensor* opt(const OptTensor& t) { return t.has_value() && t->defined() ? &*t : nullptr; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return VGO_F32;
    case at::kBFloat16: return VGO_BF16;
    case at::kHalf: return VGO_F16;
    default: TORCH_CHECK_VALUE(false, "unsupported dtype ", t);
  }
}

template <typename T = void>
T* ptr(const Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

// fp32 contiguous form of a parameter (undefined if absent).
Tensor f32(const OptTensor& t) {
  if (opt(t) == nullptr) return Tensor();
  return t->to(at::kFloat).contiguous();
}
Tensor contiguous_as(const OptTensor& t, at::ScalarType type) {
  if (opt(t) == nullptr) return Tensor();
  return t->to(type).contiguous();
}
Tensor scratch(size_t bytes, const Tensor& like) {
  return at::empty({static_cast<int64_t>((bytes + 3) / 4)}, like.options().dtype(at::kFloat));
}

// ---------------------------------------------------------------- attention ----
struct Problem {
  vgo_attn_problem p;
  Tensor q, k, v, bias;  // what p points into
};

Problem problem(const Tensor& q0, const Tensor& k0, const Tensor& v0, const OptTensor& bias0, const Tensor& out) {
  require_gpu({&q0, &k0, &v0, opt(bias0), &out});
  TORCH_CHECK_VALUE(q0.dim() == 4 && k0.dim() == 4 && v0.dim() == 4 && out.dim() == 4,
                    "q, k, v and the output must be [batch, heads, tokens, channels]");
  TORCH_CHECK_VALUE(q0.scalar_type() == k0.scalar_type() && k0.scalar_type() == v0.scalar_type() &&
                        v0.scalar_type() == out.scalar_type(),
                    "q, k, v and the output must share one dtype");
  Problem r;
  if (opt(bias0) != nullptr) {
    TORCH_CHECK_VALUE(bias0->scalar_type() == q0.scalar_type(), "the log-mass bias must be rounded to the query dtype");
    r.bias = bias0->contiguous();
  }
  const auto unit = [](const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); };
  r.q = unit(q0), r.k = unit(k0), r.v = unit(v0);
  TORCH_CHECK_VALUE(out.stride(-1) == 1, "output channel stride must be 1");
  vgo_attn_problem& p = r.p;
  p.q = ptr(r.q), p.k = ptr(r.k), p.v = ptr(r.v), p.log_mass = ptr(r.bias), p.out = ptr(out);
  p.batch = r.q.size(0), p.heads = r.q.size(1), p.n_query = r.q.size(2), p.head_dim = r.q.size(3);
  p.n_key = r.k.size(2);
  for (int i = 0; i < 3; ++i) {
    p.q_stride[i] = r.q.stride(i), p.k_stride[i] = r.k.stride(i);
    p.v_stride[i] = r.v.stride(i), p.o_stride[i] = out.stride(i);
  }
  return r;
}

// Key lengths up to this run faster on the entry without a workspace.  Measured
// on MI355X over 32,928 queries x 16 heads split into equal self-attention
// problems: at 1,029 / 1,536 / 2,058 keys the register-staged kernel takes
// 0.79 / 0.86 / 0.97 of the ping-pong kernel's time, at 3,087 / 4,116 / 8,232
// keys 1.05 / 1.08 / 1.19.  With few key tiles per 512-query task the ping-pong
// kernel's V^T pack, pipeline fill and partly empty tasks do not pay off.
constexpr int64_t kRegMaxKeys = 2560;

// split > 0: the workspace entry; 0: the entry without one; < 0: by key length, and fp32,
// which has one kernel, split over the work-groups wherever its workspace query says so.
void attention_run(const Problem& r, int64_t split) {
  const vgo_attn_problem& p = r.p;
  const int dtype = dtype_code(r.q.scalar_type());
  void* stream = stream_of(r.q);
  size_t need = 0;
  if (dtype == VGO_F32 && split != 0) {
    check(vgo_mass_bias_attn_f32_workspace(p.batch, p.heads, p.n_query, p.n_key, &need));
    const Tensor ws = need > 0 ? scratch(need, r.q) : Tensor();
    check(vgo_mass_bias_attn_f32_fwd_ws(p.q, p.k, p.v, p.log_mass, p.out, p.batch, p.heads, p.n_query, p.n_key,
                                        p.head_dim, p.q_stride, p.k_stride, p.v_stride, p.o_stride, ptr(ws), need,
                                        stream));
    return;
  }
  if (split > 0 || (split < 0 && p.n_key > kRegMaxKeys))
    check(vgo_mass_bias_attn_workspace(p.batch, p.heads, p.n_query, p.n_key, dtype, &need));
  if (need == 0) {
    check(vgo_mass_bias_attn_fwd(p.q, p.k, p.v, p.log_mass, p.out, p.batch, p.heads, p.n_query, p.n_key,
                                 p.head_dim, p.q_stride, p.k_stride, p.v_stride, p.o_stride, dtype, stream));
    return;
  }
  const Tensor ws = scratch(need, r.q);
  check(vgo_mass_bias_attn_fwd_ws(p.q, p.k, p.v, p.log_mass, p.out, p.batch, p.heads, p.n_query, p.n_key,
                                  p.head_dim, p.q_stride, p.k_stride, p.v_stride, p.o_stride, dtype, ptr(ws), need,
                                  stream));
}

void attention_into(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& bias, const Tensor& out,
                    int64_t split) {
  attention_run(problem(q, k, v, bias, out), split);
}

Tensor mass_bias_attention(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& bias) {
  Tensor out = at::empty(q.sizes(), q.options());
  attention_into(q, k, v, bias, out, -1);
  return out;
}

void attention_pair_into(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& bias, const Tensor& out,
                         const Tensor& special_q, const Tensor& special_k, const Tensor& special_v,
                         const OptTensor& special_bias, const Tensor& special_out) {
  TORCH_CHECK_VALUE(q.scalar_type() == special_q.scalar_type() && q.device() == special_q.device(),
                    "both attention problems must share one dtype and device");
  const Problem r0 = problem(q, k, v, bias, out);
  const Problem r1 = problem(special_q, special_k, special_v, special_bias, special_out);
  const int dtype = dtype_code(q.scalar_type());
  if (dtype == VGO_F32) {  // one launch each, split over the work-groups
    attention_run(r0, -1);
    attention_run(r1, -1);
    return;
  }
  const vgo_attn_problem problems[2] = {r0.p, r1.p};
  size_t need = 0;
  check(vgo_mass_bias_attn_pair_workspace(problems, 2, dtype, &need));
  const Tensor ws = need > 0 ? scratch(need, q) : Tensor();
  check(vgo_mass_bias_attn_pair_fwd_ws(problems, 2, dtype, ptr(ws), need, stream_of(q)));
}

// --------------------------------------------------------------- projection ----
void project(const Tensor& table0, const Tensor& index0, const Tensor& weight0, const OptTensor& order0,
             const Tensor& out) {
  require_gpu({&table0, &index0, &weight0, opt(order0), &out});
  TORCH_CHECK_VALUE(table0.dim() == 2 && index0.dim() == 2 && index0.size(1) == 4 && weight0.sizes() == index0.sizes(),
                    "top4_project requires table [M,D], index [N,4] and weight [N,4]");
  TORCH_CHECK_VALUE(index0.scalar_type() == at::kInt && weight0.scalar_type() == at::kFloat,
                    "top4_project requires int32 indices and float32 weights");
  const Tensor index = index0.contiguous(), weight = weight0.contiguous();
  const Tensor table = table0.stride(-1) == 1 ? table0 : table0.contiguous();
  const int64_t n = index.size(0), dim = table.size(1);
  TORCH_CHECK_VALUE(out.dim() == 2 && out.size(0) == n && out.size(1) == dim &&
                        out.scalar_type() == table.scalar_type() && out.stride(-1) == 1,
                    "top4_project output must be [N, D] of the table dtype");
  const int dtype = dtype_code(table.scalar_type());
  if (opt(order0) != nullptr) {
    TORCH_CHECK_VALUE(order0->dim() == 1 && order0->size(0) == n && order0->scalar_type() == at::kInt,
                      "top4_project order must be int32 [N]");
    const Tensor order = order0->contiguous();
    check(vgo_top4_project_ordered(ptr(table), table.stride(0), ptr<int32_t>(index), ptr<float>(weight),
                                   ptr<int32_t>(order), ptr(out), out.stride(0), n, table.size(0), dim, dtype,
                                   stream_of(table)));
    return;
  }
  check(vgo_top4_project(ptr(table), table.stride(0), ptr<int32_t>(index), ptr<float>(weight), ptr(out),
                         out.stride(0), n, table.size(0), dim, dtype, stream_of(table)));
}
void top4_project_into(const Tensor& table, const Tensor& index, const Tensor& weight, const Tensor& out) {
  project(table, index, weight, std::nullopt, out);
}
void top4_project_ordered_into(const Tensor& table, const Tensor& index, const Tensor& weight, const Tensor& order,
                               const Tensor& out) {
  project(table, index, weight, order, out);
}
Tensor top4_project(const Tensor& table, const Tensor& index, const Tensor& weight) {
  TORCH_CHECK_VALUE(table.dim() == 2 && index.dim() == 2,
                    "top4_project requires table [M,D], index [N,4] and weight [N,4]");
  Tensor out = at::empty({index.size(0), table.size(1)}, table.options());
  project(table, index, weight, std::nullopt, out);
  return out;
}

// --------------------------------------------------------------- compaction ----
// Rows, channels, token stride and head stride of a [N, C] or [H, N, 64] view.
struct Layout {
  int64_t rows, dim, token, head;
};
Layout token_layout(const Tensor& t) {
  if (t.dim() == 2) {
    TORCH_CHECK_VALUE(t.stride(1) == 1, "channel stride must be 1");
    return {t.size(0), t.size(1), t.stride(0), 64};
  }
  TORCH_CHECK_VALUE(t.dim() == 3 && t.size(-1) == 64 && t.stride(-1) == 1,
                    "compaction operands must be [N, C] or [H, N, 64] views");
  return {t.size(1), t.size(0) * 64, t.stride(1), t.stride(0)};
}

template <typename T>
const T* optional_ptr(const OptTensor& t) {
  return opt(t) == nullptr ? nullptr : static_cast<const T*>(t->data_ptr());
}

void compact_into(const Tensor& x, const Tensor& out, const OptTensor& base_rows, const Tensor& offsets,
                  int64_t segs_per_row, const OptTensor& items, int64_t item_shift, const OptTensor& item_rows,
                  const OptTensor& weights, const OptTensor& normalizer, const OptTensor& ln_weight,
                  const OptTensor& ln_bias, double ln_eps) {
  require_gpu({&x, &out, opt(base_rows), &offsets, opt(items), opt(item_rows), opt(weights), opt(normalizer)});
  const Layout xl = token_layout(x), ol = token_layout(out);
  const Tensor w = f32(ln_weight), b = w.defined() ? f32(ln_bias) : Tensor();
  check(vgo_compact(ptr(x), xl.token, xl.head, xl.rows, optional_ptr<int64_t>(base_rows), ptr<int32_t>(offsets),
                    segs_per_row, optional_ptr<uint32_t>(items), static_cast<int>(item_shift),
                    optional_ptr<int64_t>(item_rows), optional_ptr<float>(weights),
                    opt(weights) == nullptr ? 0 : weights->numel(), optional_ptr<float>(normalizer), ol.rows, ol.dim,
                    ptr<float>(w), ptr<float>(b), static_cast<float>(w.defined() ? ln_eps : 0.0), ptr(out), ol.token,
                    ol.head, dtype_code(x.scalar_type()), dtype_code(out.scalar_type()), stream_of(x)));
}

void compact_multi_into(const Tensor& x, at::IntArrayRef x_offsets, at::TensorList outs,
                        const c10::List<OptTensor>& ln_weights, const c10::List<OptTensor>& ln_biases,
                        at::ArrayRef<double> ln_eps, const OptTensor& base_rows, const Tensor& offsets,
                        int64_t segs_per_row, const OptTensor& items, int64_t item_shift, const OptTensor& item_rows,
                        const OptTensor& weights, const OptTensor& normalizer) {
  require_gpu({&x, opt(base_rows), &offsets, opt(items), opt(item_rows), opt(weights), opt(normalizer)});
  const int n = static_cast<int>(outs.size());
  TORCH_CHECK_VALUE(n >= 1 && n <= 3, "compact_multi_into: 1-3 outputs, got ", n);
  TORCH_CHECK_VALUE(x_offsets.size() == outs.size() && ln_weights.size() == outs.size() &&
                        ln_biases.size() == outs.size() && ln_eps.size() == outs.size(),
                    "compact_multi_into: one offset and LayerNorm entry per output");
  TORCH_CHECK_VALUE(x.dim() == 2 && x.stride(1) == 1,
                    "compact_multi_into: x must be an [N, W] row table with unit channel stride");
  std::array<Tensor, 6> keep;
  std::array<int64_t, 3> offs, ots, ohs;
  std::array<const float*, 3> lw{}, lb{};
  std::array<void*, 3> op{};
  int64_t rows = 0, dim = 0;
  double eps = 0.0;
  bool have_eps = false;
  for (int g = 0; g < n; ++g) {
    const Tensor& out = outs[g];
    require_gpu({&out});
    TORCH_CHECK_VALUE(out.scalar_type() == x.scalar_type(), "compact_multi_into: outputs must have x's dtype");
    const Layout l = token_layout(out);
    if (g == 0) rows = l.rows, dim = l.dim;
    TORCH_CHECK_VALUE(l.rows == rows && l.dim == dim, "compact_multi_into: every output must be ", rows, " rows x ",
                      dim, " channels, got ", l.rows, " x ", l.dim);
    TORCH_CHECK_VALUE(x_offsets[g] >= 0 && x_offsets[g] + dim <= x.size(1), "compact_multi_into: channels ",
                      x_offsets[g], "..", x_offsets[g] + dim, " lie outside x's ", x.size(1));
    offs[g] = x_offsets[g], ots[g] = l.token, ohs[g] = l.head;
    op[g] = ptr(out);
    const OptTensor w = ln_weights.get(g), b = ln_biases.get(g);
    if (opt(w) != nullptr) {
      TORCH_CHECK_VALUE(!have_eps || ln_eps[g] == eps, "compact_multi_into: the outputs' LayerNorms must share one eps");
      have_eps = true;
      eps = ln_eps[g];
      keep[2 * g] = f32(w), keep[2 * g + 1] = f32(b);
      lw[g] = ptr<float>(keep[2 * g]), lb[g] = ptr<float>(keep[2 * g + 1]);
    }
  }
  check(vgo_compact_multi(ptr(x), x.stride(0), 64, x.size(0), optional_ptr<int64_t>(base_rows),
                          ptr<int32_t>(offsets), segs_per_row, optional_ptr<uint32_t>(items),
                          static_cast<int>(item_shift), optional_ptr<int64_t>(item_rows),
                          optional_ptr<float>(weights), opt(weights) == nullptr ? 0 : weights->numel(),
                          optional_ptr<float>(normalizer), rows, dim, n, offs.data(), lw.data(), lb.data(),
                          static_cast<float>(eps), op.data(), ots.data(), ohs.data(), dtype_code(x.scalar_type()),
                          stream_of(x)));
}

// ------------------------------------------------------------ QKV epilogue ----
std::vector<Tensor> qkv_epilogue(const Tensor& qkv, int64_t heads, int64_t tokens_in, int64_t tokens_out,
                                 const OptTensor& rows0, const OptTensor& q_weight, const OptTensor& q_bias,
                                 const OptTensor& k_weight, const OptTensor& k_bias, double eps,
                                 const OptTensor& rope_sin, const OptTensor& rope_cos, int64_t rope_prefix,
                                 c10::List<bool> want, at::ScalarType out_dtype) {
  require_gpu({&qkv, opt(rows0)});
  TORCH_CHECK_VALUE(qkv.dim() == 2 && qkv.stride(1) == 1, "qkv_epilogue expects [rows, 3C] projection rows");
  TORCH_CHECK_VALUE(want.size() == 3, "qkv_epilogue: want names q, k and v");
  const Tensor rows = contiguous_as(rows0, at::kLong);
  const int64_t n_out = rows.defined() ? rows.numel() : qkv.size(0);
  TORCH_CHECK_VALUE(tokens_out > 0, "qkv_epilogue: tokens_out must be positive");
  std::vector<Tensor> outs;
  std::array<void*, 3> op{};
  for (int i = 0; i < 3; ++i) {
    const bool w = want.get(i);
    outs.push_back(w ? at::empty({n_out / tokens_out, heads, tokens_out, 64}, qkv.options().dtype(out_dtype))
                     : at::empty({0}, qkv.options().dtype(out_dtype)));
    if (w) op[i] = ptr(outs[i]);
  }
  const Tensor qw = f32(q_weight), qb = qw.defined() ? f32(q_bias) : Tensor();
  const Tensor kw = f32(k_weight), kb = kw.defined() ? f32(k_bias) : Tensor();
  const Tensor rs = f32(rope_sin), rc = rs.defined() ? f32(rope_cos) : Tensor();
  check(vgo_qkv_epilogue(ptr(qkv), qkv.stride(0), qkv.size(0), dtype_code(qkv.scalar_type()), ptr<int64_t>(rows),
                         n_out, tokens_in, tokens_out, heads, ptr<float>(qw), ptr<float>(qb), ptr<float>(kw),
                         ptr<float>(kb), static_cast<float>(eps), ptr<float>(rs), ptr<float>(rc), rope_prefix,
                         rs.defined() ? rs.size(0) : 0, op[0], op[1], op[2], dtype_code(out_dtype), stream_of(qkv)));
  return outs;
}

// ------------------------------------------------------------ residual rows ----
std::vector<Tensor> residual_layer_norm(const Tensor& x, const OptTensor& branch, const OptTensor& gamma,
                                        const OptTensor& ln_weight, const OptTensor& ln_bias, double eps,
                                        bool has_norm, bool write_sum, std::optional<at::ScalarType> norm_dtype,
                                        bool norm_f32, double unit_eps) {
  require_gpu({&x, opt(branch), opt(gamma), opt(ln_weight), opt(ln_bias)});
  TORCH_CHECK_VALUE(x.scalar_type() == at::kFloat, "residual_layer_norm: x must be float32");
  TORCH_CHECK_VALUE(x.dim() >= 1, "residual_layer_norm: x must be [..., dim]");
  const int64_t dim = x.size(-1);
  const Tensor rows = x.reshape({-1, dim});
  Tensor b_rows;
  if (opt(branch) != nullptr) {
    TORCH_CHECK_VALUE(branch->sizes() == x.sizes(), "residual_layer_norm: branch ", branch->sizes(), " != x ", x.sizes());
    b_rows = branch->reshape({-1, dim});
  }
  const auto make = [&](bool wanted, at::ScalarType type) {
    return wanted ? at::empty(x.sizes(), x.options().dtype(type)) : Tensor();
  };
  const bool cast = has_norm && norm_dtype.has_value();
  const Tensor total = make(write_sum && b_rows.defined(), at::kFloat);
  const Tensor normed = make(cast, norm_dtype.value_or(at::kBFloat16));
  const Tensor normed32 = make(has_norm && norm_f32, at::kFloat);
  TORCH_CHECK_VALUE(unit_eps < 0 || cast, "residual_layer_norm: unit rows need a norm and norm_dtype");
  const Tensor unit = make(unit_eps >= 0, norm_dtype.value_or(at::kBFloat16));
  const Tensor w = has_norm ? f32(ln_weight) : Tensor(), b = has_norm ? f32(ln_bias) : Tensor();
  const Tensor g = f32(gamma);
  check(vgo_residual_layer_norm(
      ptr<float>(rows), rows.stride(0), ptr(b_rows), b_rows.defined() ? b_rows.stride(0) : 0,
      b_rows.defined() ? dtype_code(b_rows.scalar_type()) : VGO_F32, ptr<float>(g), ptr<float>(w), ptr<float>(b),
      static_cast<float>(has_norm ? eps : 0.0), rows.size(0), dim, ptr<float>(total), dim, ptr(normed), dim,
      normed.defined() ? dtype_code(normed.scalar_type()) : VGO_BF16, ptr<float>(normed32), dim, ptr(unit), dim,
      static_cast<float>(unit_eps >= 0 ? unit_eps : 0.0), stream_of(x)));
  const auto or_empty = [&](const Tensor& t) { return t.defined() ? t : at::empty({0}, x.options()); };
  return {or_empty(total), or_empty(normed), or_empty(normed32), or_empty(unit)};
}

std::vector<Tensor> restore_residual_layer_norm(const Tensor& x, const Tensor& table0, const Tensor& index0,
                                                const OptTensor& weight0, const OptTensor& gamma,
                                                const OptTensor& ln_weight, const OptTensor& ln_bias, double eps,
                                                at::ScalarType norm_dtype) {
  require_gpu({&x, &table0, &index0, opt(weight0), opt(gamma), opt(ln_weight), opt(ln_bias)});
  TORCH_CHECK_VALUE(x.scalar_type() == at::kFloat, "restore_residual_layer_norm: x must be float32");
  TORCH_CHECK_VALUE(x.dim() >= 1, "restore_residual_layer_norm: x must be [..., dim]");
  const int64_t dim = x.size(-1);
  const Tensor rows = x.reshape({-1, dim});
  const int64_t n = rows.size(0);
  TORCH_CHECK_VALUE(table0.dim() == 2 && table0.size(1) == dim, "restore_residual_layer_norm: table ", table0.sizes(),
                    " must be [M, ", dim, "]");
  if (opt(weight0) == nullptr) {
    TORCH_CHECK_VALUE(index0.dim() == 1 && index0.size(0) == n,
                      "restore_residual_layer_norm: a one-hot index must be [rows]");
  } else {
    TORCH_CHECK_VALUE(index0.dim() == 2 && index0.size(0) == n && index0.size(1) == 4 &&
                          weight0->sizes() == index0.sizes(),
                      "restore_residual_layer_norm: index and weight must be [rows, 4]");
  }
  TORCH_CHECK_VALUE(index0.scalar_type() == at::kInt &&
                        (opt(weight0) == nullptr || weight0->scalar_type() == at::kFloat),
                    "restore_residual_layer_norm: int32 indices and float32 weights");
  TORCH_CHECK_VALUE(norm_dtype == at::kBFloat16 || norm_dtype == at::kHalf,
                    "restore_residual_layer_norm: norm_dtype must be bfloat16 or float16");
  const Tensor index = index0.contiguous();
  const Tensor weight = opt(weight0) == nullptr ? Tensor() : weight0->contiguous();
  const Tensor table = table0.stride(-1) == 1 ? table0 : table0.contiguous();
  const Tensor w = f32(ln_weight), b = f32(ln_bias), g = f32(gamma);
  Tensor total = at::empty(x.sizes(), x.options());
  Tensor normed = at::empty(x.sizes(), x.options().dtype(norm_dtype));
  check(vgo_restore_residual_layer_norm(
      ptr<float>(rows), rows.stride(0), ptr(table), table.stride(0), table.size(0), dtype_code(table.scalar_type()),
      ptr<int32_t>(index), ptr<float>(weight), ptr<float>(g), ptr<float>(w), ptr<float>(b), static_cast<float>(eps),
      n, dim, ptr<float>(total), dim, ptr(normed), dim, dtype_code(norm_dtype), stream_of(x)));
  return {total, normed};
}

// -------------------------------------------------------------- whole blocks ----
// Exact GELU of a tensor that nothing else holds.  From 2^23 bf16 values on the table kernel runs in
// place, with the bits of torch's kernel (us, torch / table: 2^22 values 6.6 / 8.5, 2^23 10.2 / 9.1,
// 2^25 29.7 / 23.0, 32,928 x 4,096 122 / 107): below, its table costs more than it saves.
Tensor gelu_owned(const Tensor& t) {
  if (t.scalar_type() != at::kBFloat16 || t.numel() < (int64_t{1} << 23) || !t.is_contiguous() ||
      reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0)
    return at::gelu(t);
  check(vgo_gelu_bf16(ptr(t), ptr(t), t.numel(), stream_of(t)));
  return t;
}

// x + gamma2 * fc2(gelu(fc1(h))): a block's MLP and its last residual pass, the
// Linears in h's dtype (parameters already cast to it), as block.py:126-127 under autocast.
Tensor mlp_tail(const Tensor& x, const Tensor& h, const Tensor& fc1_w, const OptTensor& fc1_b, const Tensor& fc2_w,
                const OptTensor& fc2_b, const OptTensor& gamma) {
  const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
  const Tensor y = at::linear(gelu_owned(at::linear(h, fc1_w, fc1_b)), fc2_w, fc2_b);
  return residual_layer_norm(x, y.reshape(x.sizes()), gamma, std::nullopt, std::nullopt, 0.0, false, true,
                             std::nullopt, false, -1.0)[0];
}

// An unmerged block (block.py:89-129 at inference under bf16 / f16 autocast) on an fp32 stream
// x [B, N, C]: norm1, qkv, the q/k LayerNorm + RoPE epilogue, attention, the output projection,
// residual + norm2, and mlp_tail.  `norms`: norm1 weight, bias, norm2 weight, bias, then the q and
// k LayerNorms' weight, bias (absent ones None); `linears`: qkv, proj, fc1, fc2 weight and bias
// in `dtype`; `gammas`: the two LayerScales'.
Tensor dense_block(const Tensor& x, const c10::List<OptTensor>& norms, at::ArrayRef<double> eps,
                   const c10::List<OptTensor>& linears, const c10::List<OptTensor>& gammas, int64_t heads,
                   const OptTensor& rope_sin, const OptTensor& rope_cos, at::ScalarType dtype) {
  TORCH_CHECK_VALUE(x.dim() == 3 && norms.size() == 8 && eps.size() == 3 && linears.size() == 8 && gammas.size() == 2,
                    "dense_block: x [B, N, C], 8 norm, 3 eps, 8 linear and 2 gamma entries");
  const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
  const int64_t batch = x.size(0), tokens = x.size(1), dim = x.size(2);
  const auto linear = [&](const Tensor& in, int i) { return at::linear(in, *linears.get(2 * i), linears.get(2 * i + 1)); };
  // In a scope of its own: the packed rows, q, k and the attention's output are free again in the MLP.
  const std::vector<Tensor> rows = [&] {
    const Tensor h = residual_layer_norm(x, std::nullopt, std::nullopt, norms.get(0), norms.get(1), eps[0], true, true,
                                         dtype, false, -1.0)[1];
    const Tensor qkv = linear(h, 0);
    const int64_t prefix = opt(rope_sin) == nullptr ? 0 : tokens - rope_sin->size(-2);
    TORCH_CHECK(prefix >= 0, "dense_block: more RoPE positions than tokens");
    // The attention takes v where the projection wrote it: copying it head-major was a third of
    // the epilogue's bytes (a block of 32 x 1,029 tokens 1,384 -> 1,370 us).  Copied only where the
    // kernels' 32-bit token offsets (stride x tokens < 2^31) do not reach; layers.py `_value_rows`
    // is the same rule.
    const bool v_in_place = tokens * 3 * dim < (int64_t{1} << 31);
    const std::vector<Tensor> heads_out =
        qkv_epilogue(qkv.reshape({batch * tokens, 3 * dim}), heads, tokens, tokens, std::nullopt, norms.get(4),
                     norms.get(5), norms.get(6), norms.get(7), eps[2], rope_sin, rope_cos, prefix,
                     c10::List<bool>({true, true, !v_in_place}), dtype);
    const Tensor v = v_in_place ? qkv.view({batch, tokens, 3, heads, 64}).select(2, 2).transpose(1, 2) : heads_out[2];
    const Tensor attended = at::empty({batch, tokens, heads, 64}, x.options().dtype(dtype));
    attention_into(heads_out[0], heads_out[1], v, std::nullopt, attended.permute({0, 2, 1, 3}), -1);
    return residual_layer_norm(x, linear(attended.view({batch, tokens, dim}), 1), gammas.get(0), norms.get(2),
                               norms.get(3), eps[1], true, true, dtype, false, -1.0);
  }();
  return mlp_tail(rows[0], rows[1], *linears.get(4), linears.get(5), *linears.get(6), linears.get(7), gammas.get(1));
}

// ------------------------------------------------------------------- plans ----
Tensor normalize_rows(const Tensor& x0, const OptTensor& rows0, double eps, at::ScalarType out_dtype) {
  require_gpu({&x0, opt(rows0)});
  const Tensor x = x0.dim() == 2 && x0.stride(-1) == 1 ? x0 : x0.reshape({-1, x0.size(-1)}).contiguous();
  const Tensor rows = contiguous_as(rows0, at::kLong);
  const int64_t n = rows.defined() ? rows.numel() : x.size(0);
  Tensor out = at::empty({n, x.size(1)}, x.options().dtype(out_dtype));
  check(vgo_normalize_rows(ptr(x), x.stride(0), x.size(0), dtype_code(x.scalar_type()), ptr<int64_t>(rows), n,
                           x.size(1), static_cast<float>(eps), ptr(out), out.stride(0), dtype_code(out_dtype),
                           stream_of(x)));
  return out;
}

std::tuple<Tensor, Tensor> csr_build(const Tensor& keys0, int64_t n_buckets) {
  require_gpu({&keys0});
  const Tensor keys = keys0.to(at::kInt).contiguous();
  const int64_t n = keys.numel();
  size_t need = 0;
  check(vgo_csr_workspace(n, n_buckets, &need));
  const Tensor ws = at::empty({static_cast<int64_t>(need) + 256}, keys.options().dtype(at::kByte));
  char* base = ptr<char>(ws);
  base += (256 - reinterpret_cast<uintptr_t>(base) % 256) % 256;
  Tensor order = at::empty({n}, keys.options()), offsets = at::empty({n_buckets + 1}, keys.options());
  check(vgo_csr_build(ptr<uint32_t>(keys), n, n_buckets, base, need, ptr<uint32_t>(order), ptr<int32_t>(offsets),
                      stream_of(keys)));
  return {order, offsets};
}

std::tuple<Tensor, Tensor> corner_csr(const Tensor& parent0, int64_t n_dest) {
  require_gpu({&parent0});
  const int64_t corners = parent0.size(-1), n = parent0.numel();
  const Tensor parent = parent0.to(at::kLong).contiguous();
  const auto options = parent.options().dtype(at::kInt);
  size_t need = 0;
  check(vgo_csr_workspace(n, n_dest * corners, &need));
  const Tensor ws = at::empty({static_cast<int64_t>(need) + 256}, options.dtype(at::kByte));
  char* base = ptr<char>(ws);
  base += (256 - reinterpret_cast<uintptr_t>(base) % 256) % 256;
  Tensor order = at::empty({n}, options), offsets = at::empty({n_dest * corners + 1}, options);
  check(vgo_corner_csr(ptr<int64_t>(parent), n, corners, n_dest, base, need, ptr<uint32_t>(order),
                       ptr<int32_t>(offsets), stream_of(parent)));
  return {order, offsets};
}

std::tuple<Tensor, Tensor> segment_mass(const Tensor& offsets, int64_t segs_per_row, const Tensor& order,
                                        const OptTensor& weights0, int64_t rows, double start, bool want_log) {
  require_gpu({&offsets, &order, opt(weights0)});
  const Tensor weights = f32(weights0);
  const auto options = offsets.options().dtype(at::kFloat);
  Tensor mass = at::empty({rows}, options), log_mass = at::empty({want_log ? rows : 0}, options);
  check(vgo_segment_mass(ptr<int32_t>(offsets), segs_per_row, ptr<uint32_t>(order), ptr<float>(weights),
                         weights.defined() ? weights.numel() : 0, rows, static_cast<float>(start), ptr<float>(mass),
                         want_log ? ptr<float>(log_mass) : nullptr, stream_of(offsets)));
  return {mass, log_mass};
}

// Top-K bf16 cosine matches of every source row; index (and values, where given) are
// written.  n_src < 0: every row of src (or of src_rows).
void similarity_topk(const Tensor& src0, const Tensor& dict0, int64_t topk, const OptTensor& src_rows0,
                     const OptTensor& n_src_device, int64_t n_src, int64_t n0, int64_t off1, int64_t n_dict,
                     const OptTensor& index_map0, const OptTensor& values, const Tensor& index,
                     const OptTensor& scores) {
  require_gpu({&src0, &dict0, opt(src_rows0), opt(n_src_device), opt(index_map0), opt(values), &index, opt(scores)});
  TORCH_CHECK_VALUE(src0.scalar_type() == at::kBFloat16 && dict0.scalar_type() == at::kBFloat16 && src0.dim() == 2 &&
                        dict0.dim() == 2,
                    "similarity_topk expects bf16 operands");
  const Tensor src = src0.stride(-1) == 1 ? src0 : src0.contiguous();
  const Tensor dict = dict0.stride(-1) == 1 ? dict0 : dict0.contiguous();
  const Tensor src_rows = contiguous_as(src_rows0, at::kLong), index_map = contiguous_as(index_map0, at::kLong);
  if (n_src < 0) n_src = src_rows.defined() ? src_rows.numel() : src.size(0);
  const auto shaped = [&](const Tensor& t) {
    return t.dim() == 2 && t.size(0) == n_src && t.size(1) == topk && t.is_contiguous();
  };
  TORCH_CHECK_VALUE(shaped(index) && (index.scalar_type() == at::kLong || index.scalar_type() == at::kInt) &&
                        (opt(values) == nullptr || (shaped(*values) && values->scalar_type() == at::kFloat)),
                    "similarity_topk: `out` must be contiguous [n, K] fp32 values and indices");
  int parts = 0;
  size_t need = 0;
  check(vgo_similarity_topk_workspace(n_src, n_dict, static_cast<int>(topk), &parts, &need));
  const Tensor ws = at::empty({std::max<int64_t>(1, static_cast<int64_t>(need / 8))}, src.options().dtype(at::kLong));
  const bool wide = index.scalar_type() == at::kLong;
  check(vgo_similarity_topk(
      ptr(src), src.stride(0), src.size(0), ptr<int64_t>(src_rows), optional_ptr<int>(n_src_device), n_src, ptr(dict),
      dict.stride(0), dict.size(0), n0, off1, n_dict, src.size(1), static_cast<int>(topk), ptr(ws), ws.numel() * 8,
      opt(values) == nullptr ? nullptr : ptr<float>(*values), wide ? ptr<int64_t>(index) : nullptr,
      wide ? nullptr : ptr<int32_t>(index), ptr<int64_t>(index_map), opt(scores) == nullptr ? nullptr : ptr(*scores),
      opt(scores) == nullptr ? 0 : scores->stride(0), stream_of(src)));
}

// The FastVGGT match of tokens [B, N, C]: every source's best destination (fp32 score, int32
// position), from the tokens' normalised rows or from bf16 unit rows as given.
std::tuple<Tensor, Tensor> fastvggt_match(const Tensor& tokens, const Tensor& sources, const Tensor& destinations,
                                          bool prenormalized) {
  require_gpu({&tokens, &sources, &destinations});
  TORCH_CHECK_VALUE(tokens.dim() == 3, "FastVGGT tokens must be [batch, tokens, channels]");
  TORCH_CHECK_VALUE(!prenormalized || tokens.scalar_type() == at::kBFloat16,
                    "prenormalized FastVGGT tokens must be bf16 unit rows");
  const int64_t batch = tokens.size(0), n = sources.numel(), n_dict = destinations.numel();
  Tensor best = at::empty({batch, n}, tokens.options().dtype(at::kFloat));
  Tensor target = at::empty({batch, n}, tokens.options().dtype(at::kInt));
  for (int64_t b = 0; b < batch; ++b) {
    const Tensor row = tokens.select(0, b), x = row.stride(-1) == 1 ? row : row.contiguous();
    const Tensor src = prenormalized ? x : normalize_rows(x, sources, 1e-12, at::kBFloat16);
    const Tensor dst =
        prenormalized ? x.index_select(0, destinations) : normalize_rows(x, destinations, 1e-12, at::kBFloat16);
    similarity_topk(src, dst, 1, prenormalized ? OptTensor(sources) : std::nullopt, std::nullopt, -1, n_dict, 0,
                    n_dict, std::nullopt, best.select(0, b).view({n, 1}), target.select(0, b).view({n, 1}),
                    std::nullopt);
  }
  return {best, target};
}

std::tuple<Tensor, Tensor, Tensor> fastvggt_assemble(const Tensor& best, const Tensor& target, const Tensor& sources,
                                                     const Tensor& destinations, int64_t total, int64_t removed) {
  require_gpu({&best, &target, &sources, &destinations});
  const int64_t batch = best.size(0), n_src = sources.numel();
  TORCH_CHECK_VALUE(best.is_contiguous() && target.is_contiguous() && sources.is_contiguous() &&
                        destinations.is_contiguous() && best.scalar_type() == at::kFloat &&
                        target.scalar_type() == at::kInt && sources.scalar_type() == at::kLong &&
                        destinations.scalar_type() == at::kLong && best.numel() == batch * n_src &&
                        target.numel() == batch * n_src,
                    "fastvggt_assemble: contiguous fp32 scores and int32 targets [B, n], int64 ids");
  const auto options = sources.options();
  Tensor keep = at::empty({batch, total - removed}, options), inverse = at::empty({batch, total}, options);
  Tensor flags = at::empty({batch, n_src}, options.dtype(at::kByte));
  size_t need = 0;
  check(vgo_fastvggt_assemble_workspace(batch, n_src, total, &need));
  const Tensor ws = scratch(need, best);
  check(vgo_fastvggt_assemble_ws(ptr<float>(best), ptr<int32_t>(target), ptr<int64_t>(sources),
                                 ptr<int64_t>(destinations), batch, n_src, destinations.numel(), total, removed,
                                 ptr<int64_t>(keep), ptr<int64_t>(inverse), ptr<uint8_t>(flags), ptr(ws), need,
                                 stream_of(best)));
  return {keep, inverse, flags};
}

// fastvggt_assemble of one batch element with its clusters' CSR, sizes and log sizes from one
// launch: (keep, inverse, flags, inverse as int32, order, offsets, mass, log_mass).
std::vector<Tensor> fastvggt_plan(const Tensor& best, const Tensor& target, const Tensor& sources,
                                  const Tensor& destinations, int64_t total, int64_t removed) {
  require_gpu({&best, &target, &sources, &destinations});
  const int64_t n_src = sources.numel(), kept = total - removed;
  TORCH_CHECK_VALUE(best.is_contiguous() && target.is_contiguous() && sources.is_contiguous() &&
                        destinations.is_contiguous() && best.scalar_type() == at::kFloat &&
                        target.scalar_type() == at::kInt && sources.scalar_type() == at::kLong &&
                        destinations.scalar_type() == at::kLong && best.numel() == n_src && target.numel() == n_src &&
                        kept >= 0,
                    "fastvggt_plan: contiguous fp32 scores and int32 targets [1, n], int64 ids");
  const auto ids = sources.options(), i32 = ids.dtype(at::kInt), f32s = ids.dtype(at::kFloat);
  std::vector<Tensor> r = {at::empty({1, kept}, ids),   at::empty({1, total}, ids), at::empty({1, n_src}, ids.dtype(at::kByte)),
                           at::empty({total}, i32),     at::empty({total}, i32),    at::empty({kept + 1}, i32),
                           at::empty({kept}, f32s),     at::empty({kept}, f32s)};
  check(vgo_fastvggt_plan(ptr<float>(best), ptr<int32_t>(target), ptr<int64_t>(sources), ptr<int64_t>(destinations),
                          n_src, destinations.numel(), total, removed, ptr<int64_t>(r[0]), ptr<int64_t>(r[1]),
                          ptr<int32_t>(r[3]), ptr<uint8_t>(r[2]), ptr<uint32_t>(r[4]), ptr<int32_t>(r[5]),
                          ptr<float>(r[6]), ptr<float>(r[7]), stream_of(best)));
  return r;
}

// A merged block (block.py:219-226 under bf16 / f16 autocast) on an fp32 stream x [1, N, C] with a
// token plan: norm1 and the qkv projection unless given, compaction of the clusters (offsets,
// order, counts, contribution), mass-bias attention, the output projection, restore (inverse)
// + residual + norm2 in one pass, and mlp_tail.  Parameters as dense_block's.
Tensor merged_block(const Tensor& x, const OptTensor& h0, const OptTensor& qkv0, const Tensor& offsets,
                    const Tensor& order, const Tensor& counts, const OptTensor& contribution, const Tensor& inverse,
                    const OptTensor& log_mass, const c10::List<OptTensor>& norms, at::ArrayRef<double> eps,
                    const c10::List<OptTensor>& linears, const c10::List<OptTensor>& gammas, int64_t heads,
                    at::ScalarType dtype) {
  TORCH_CHECK_VALUE(x.dim() == 3 && x.size(0) == 1 && norms.size() == 8 && eps.size() == 3 && linears.size() == 8 &&
                        gammas.size() == 2,
                    "merged_block: x [1, N, C], 8 norm, 3 eps, 8 linear and 2 gamma entries");
  const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
  const int64_t tokens = x.size(1), dim = x.size(2), kept = counts.numel();
  const auto linear = [&](const Tensor& in, int i) { return at::linear(in, *linears.get(2 * i), linears.get(2 * i + 1)); };
  const std::vector<Tensor> rows = [&] {  // (a scope of its own, as dense_block's)
    Tensor qkv = opt(qkv0) == nullptr ? Tensor() : *qkv0;
    if (!qkv.defined()) {
      const Tensor h = opt(h0) != nullptr ? *h0
                                          : residual_layer_norm(x, std::nullopt, std::nullopt, norms.get(0),
                                                                norms.get(1), eps[0], true, true, dtype, false, -1.0)[1];
      qkv = linear(h, 0);
    }
    const Tensor operands = at::empty({3, 1, heads, kept, 64}, x.options().dtype(dtype));
    const Tensor q = operands.select(0, 0), k = operands.select(0, 1), v = operands.select(0, 2);
    const std::array<Tensor, 3> outs = {q.select(0, 0), k.select(0, 0), v.select(0, 0)};
    const std::array<int64_t, 3> at_channel = {0, dim, 2 * dim};
    const std::array<double, 3> ln_eps = {eps[2], eps[2], 0.0};
    const c10::List<OptTensor> weights({norms.get(4), norms.get(6), std::nullopt});
    const c10::List<OptTensor> biases({norms.get(5), norms.get(7), std::nullopt});
    compact_multi_into(qkv.reshape({tokens, 3 * dim}), at_channel, outs, weights, biases, ln_eps, std::nullopt, offsets,
                       1, order, 0, std::nullopt, contribution, counts);
    OptTensor bias;
    if (opt(log_mass) != nullptr) bias = log_mass->reshape({-1}).to(dtype);
    const Tensor attended = at::empty({1, kept, heads, 64}, x.options().dtype(dtype));
    attention_into(q, k, v, bias, attended.permute({0, 2, 1, 3}), -1);
    const Tensor table = linear(attended.view({kept, dim}), 1);
    return restore_residual_layer_norm(x, table, inverse, std::nullopt, gammas.get(0), norms.get(2), norms.get(3),
                                       eps[1], dtype);
  }();
  return mlp_tail(rows[0], rows[1], *linears.get(4), linears.get(5), *linears.get(6), linears.get(7), gammas.get(1));
}

// sin and cos tables into two contiguous fp32 [h * w, head_dim].
void rope_table(const Tensor& sin, const Tensor& cos, int64_t h, int64_t w, double base) {
  require_gpu({&sin, &cos});
  for (const Tensor* t : {&sin, &cos})
    TORCH_CHECK(t->dim() == 2 && t->size(0) == h * w && t->sizes() == sin.sizes() && t->device() == sin.device() &&
                    t->scalar_type() == at::kFloat && t->is_contiguous(),
                "rope_table: sin and cos must be contiguous float32 [h * w, head_dim]");
  check(vgo_rope_table(h, w, sin.size(1), static_cast<float>(base), ptr<float>(sin), ptr<float>(cos), stream_of(sin)));
}

// Operators by what autograd makes of them.  Path: gradient-free, but part of a recorded graph, whose
// backward raises; a tensor's tangents end there.  Plan: read their inputs' values alone, as a plan does.
// Blocks: likewise, whole sequences of launches that only plain tensors reach.
constexpr const char* kPath[] = {"mass_bias_attention", "top4_project", "qkv_epilogue", "residual_layer_norm",
                                 "restore_residual_layer_norm"};
constexpr const char* kBlocks[] = {"mlp_tail", "dense_block", "merged_block"};
constexpr const char* kPathInto[] = {"attention_into", "attention_pair_into", "top4_project_into",
                                     "top4_project_ordered_into", "compact_into", "compact_multi_into"};
constexpr const char* kPlan[] = {"normalize_rows", "csr_build", "corner_csr", "segment_mass", "fastvggt_assemble",
                                 "fastvggt_match", "fastvggt_plan"};
constexpr const char* kPlanInto[] = {"similarity_topk", "rope_table"};

template <typename Visit>
void each_tensor(const c10::IValue& value, Visit visit) {
  if (value.isTensor()) {
    if (value.toTensor().defined()) visit(value.toTensor());
  } else if (value.isList()) {
    for (const c10::IValue& item : value.toListRef()) each_tensor(item, visit);
  }
}

// Autograd key.  History: where an input requires grad (and grad mode is on) floating outputs do too,
// with a backward that raises; written tensors are left as they are.
template <bool kHistory>
void autograd(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const size_t arguments = op.schema().arguments().size(), returns = op.schema().returns().size();
  torch::autograd::edge_list inputs;
  if constexpr (kHistory) {
    if (at::GradMode::is_enabled()) {
      bool tangent = false;
      for (const c10::IValue& value : torch::jit::last(*stack, arguments))
        each_tensor(value, [&](const Tensor& t) {
          if (t.requires_grad()) inputs.push_back(torch::autograd::impl::gradient_edge(t));
          tangent |= t._fw_grad(/*level=*/0).defined();
        });
      TORCH_CHECK_NOT_IMPLEMENTED(inputs.empty() || !tangent, op.operator_name().name,
                                  " has no derivative: tensors that require grad cannot carry tangents through it");
    }
  }
  {
    const at::AutoDispatchBelowAutograd below;
    op.redispatchBoxed(keys & c10::after_autograd_keyset, stack);
  }
  if (inputs.empty()) return;
  const std::shared_ptr<torch::autograd::Node> node(
      new torch::autograd::NotImplemented(op.operator_name().name, std::move(inputs)), torch::autograd::deleteNode);
  for (const c10::IValue& value : torch::jit::last(*stack, returns))
    each_tensor(value, [&](const Tensor& t) {
      if (torch::autograd::isDifferentiableType(t.scalar_type())) torch::autograd::set_history(t, node);
    });
}

// ADInplaceOrView key of operators that write arguments: their versions count the write.
void written(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  std::vector<Tensor> outputs;
  const auto& arguments = op.schema().arguments();
  const auto values = torch::jit::last(*stack, arguments.size());
  for (size_t i = 0; i < arguments.size(); ++i)
    if (arguments[i].alias_info() != nullptr && arguments[i].alias_info()->isWrite())
      each_tensor(values[i], [&](const Tensor& t) { outputs.push_back(t); });
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    op.redispatchBoxed(keys & c10::after_ADInplaceOrView_keyset, stack);
  }
  for (const Tensor& t : outputs)
    if (!t.is_inference()) torch::autograd::impl::bump_version(t);
}

// vmap over a planner's or a block's operator: refused.  The path's operators take torch's fallback,
// which runs one call per batch element where the results are new tensors.
void no_batching(const c10::OperatorHandle& op, c10::DispatchKeySet, torch::jit::Stack*) {
  TORCH_CHECK(false, op.operator_name().name, " has no batching rule (vmap)");
}

// `fn` with its first argument's device as the current device.  The kernels' launches, the device
// properties that size them and static scratch all go by the current device, and torch's default
// stream of any device is the null stream, that is, the current device's.
template <auto fn>
struct OnDevice;
template <typename R, typename... Rest, R (*fn)(const Tensor&, Rest...)>
struct OnDevice<fn> {
  static R call(const Tensor& first, Rest... rest) {
    c10::OptionalDeviceGuard guard;
    if (first.is_cuda()) guard.reset_device(first.device());
    return fn(first, std::forward<Rest>(rest)...);
  }
};
template <auto fn>
constexpr auto on_device = &OnDevice<fn>::call;

void register_cuda(torch::Library& m) {
  m.impl("mass_bias_attention", on_device<mass_bias_attention>);
  m.impl("attention_into", on_device<attention_into>);
  m.impl("attention_pair_into", on_device<attention_pair_into>);
  m.impl("top4_project", on_device<top4_project>);
  m.impl("top4_project_into", on_device<top4_project_into>);
  m.impl("top4_project_ordered_into", on_device<top4_project_ordered_into>);
  m.impl("compact_into", on_device<compact_into>);
  m.impl("compact_multi_into", on_device<compact_multi_into>);
  m.impl("qkv_epilogue", on_device<qkv_epilogue>);
  m.impl("residual_layer_norm", on_device<residual_layer_norm>);
  m.impl("restore_residual_layer_norm", on_device<restore_residual_layer_norm>);
  m.impl("mlp_tail", on_device<mlp_tail>);
  m.impl("dense_block", on_device<dense_block>);
  m.impl("normalize_rows", on_device<normalize_rows>);
  m.impl("rope_table", on_device<rope_table>);
  m.impl("csr_build", on_device<csr_build>);
  m.impl("corner_csr", on_device<corner_csr>);
  m.impl("segment_mass", on_device<segment_mass>);
  m.impl("fastvggt_assemble", on_device<fastvggt_assemble>);
  m.impl("fastvggt_match", on_device<fastvggt_match>);
  m.impl("fastvggt_plan", on_device<fastvggt_plan>);
  m.impl("similarity_topk", on_device<similarity_topk>);
  m.impl("merged_block", on_device<merged_block>);
}

void register_autograd(torch::Library& m) {
  for (const char* name : kPath) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd<true>>());
  for (const char* name : kPathInto) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd<true>>());
  for (const char* name : kBlocks) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd<true>>());
  for (const char* name : kPlan) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd<false>>());
  for (const char* name : kPlanInto) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd<false>>());
}

void register_inplace(torch::Library& m) {
  for (const char* name : kPathInto) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&written>());
  for (const char* name : kPlanInto) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&written>());
}

void register_batched(torch::Library& m) {
  const auto refuse = [&](const auto& names) {
    for (const char* name : names) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&no_batching>());
  };
  refuse(kBlocks), refuse(kPlan), refuse(kPlanInto);
}

}  // namespace

// Registers the implementations with the schemas that ops.py defined; null, or what is wrong (the
// text stays valid), with nothing registered.  A call and not the initialisers of TORCH_LIBRARY_IMPL:
// an exception there, as where the library was built for other schemas, ends the process that loads it.
extern "C" __attribute__((visibility("default"))) const char* vgo_torch_register() {
  static std::string message;
  try {
    std::vector<std::unique_ptr<torch::Library>> libraries;
    const auto add = [&](c10::DispatchKey key, void (*fill)(torch::Library&)) {
      libraries.push_back(std::make_unique<torch::Library>(torch::Library::IMPL, "vgo", key, __FILE__, __LINE__));
      fill(*libraries.back());
    };
    add(c10::DispatchKey::CUDA, register_cuda);
    add(c10::DispatchKey::Autograd, register_autograd);
    add(c10::DispatchKey::ADInplaceOrView, register_inplace);
    add(c10::DispatchKey::FuncTorchBatched, register_batched);
    for (auto& library : libraries) (void)library.release();  // they last as long as the process
    return nullptr;
  } catch (const c10::Error& error) {
    message = error.what_without_backtrace();
  } catch (const std::exception& error) {
    message = error.what();
  }
  return message.c_str();
}
