"""torch.library operators of the merged global-attention path (namespace `vgo`).

Every kernel a merged block launches is a `torch.ops.vgo.*` operator, so the
dispatcher, `torch.compile` and fake-tensor tracing see them as single ops:

* `vgo::mass_bias_attention(q, k, v, log_key_mass?) -> Tensor`  -- the reference's
  operator (vggt_omega/models/mass_bias_attention.py:85-129) on already-cast
  inputs; `vgo::attention_into` / `vgo::attention_pair_into` write into given
  (strided) outputs, the pair form also running the dense special-query pass of
  vggt_omega/models/layers/attention.py:406-422 in the same launch;
* `vgo::top4_project(table, index, weight) -> Tensor`, `vgo::top4_project_into` and
  `vgo::top4_project_ordered_into` -- the plans' restore (token_merging.py:387-414,
  193-196);
* `vgo::compact_into`, `vgo::compact_multi_into` -- Q/K/V compaction
  (token_merging.py:343-385, 176-191) with the q/k LayerNorm fused;
* `vgo::qkv_epilogue` -- the packed projection split into head-major q/k/v with
  LayerNorm64 and RoPE (layers/attention.py:243-262, 334-341);
* `vgo::residual_layer_norm` -- LayerScale, residual add, LayerNorm and the
  autocast cast of a block (layers/block.py:126-127, 219-226);
  `vgo::restore_residual_layer_norm` -- the same with the plan restore
  (token_merging.py:387-414, 193-196) computed in the pass.

* `vgo::mlp_tail`, `vgo::dense_block`, `vgo::merged_block` -- a block's MLP with its
  last residual pass, a whole unmerged block (layers/block.py:89-129) and a whole
  merged block over a token plan (:219-226), for eager inference; and the plan
  builders' kernels (`vgo::normalize_rows`, `similarity_topk`, `fastvggt_match`,
  `fastvggt_assemble`, `fastvggt_plan`, `csr_build`, `corner_csr`,
  `segment_mass`).

The CUDA (HIP) implementations are native (csrc/torch_ops.cpp, built into
`libvgo_ops.so`) and call `libvgo.so` through its C ABI.  The operators a
traced graph can hold have fake implementations that only describe their
outputs; the block sequences, which tracing never takes, have none.  There is no
CPU implementation: CPU tensors fail in the dispatcher.
"""
import torch

from . import _lib

_SCHEMAS = (
    # softmax(q k^T / 8 + log_key_mass) v for [B, H, N, 64] q/k/v of one dtype; the bias
    # already rounded to that dtype (or None); a new contiguous output.
    "mass_bias_attention(Tensor q, Tensor k, Tensor v, Tensor? log_key_mass) -> Tensor",
    # The same into `out` (any strides with a unit channel stride); split: -1 picks the
    # entry by key length, 0 the entry without a workspace, 1 the workspace entry.
    "attention_into(Tensor q, Tensor k, Tensor v, Tensor? bias, Tensor(a!) out, SymInt split) -> ()",
    # Merged attention and the dense special-query pass: one launch in bf16 / f16, in fp32 one
    # after the other.
    "attention_pair_into(Tensor q, Tensor k, Tensor v, Tensor? bias, Tensor(a!) out, Tensor special_q, "
    "Tensor special_k, Tensor special_v, Tensor? special_bias, Tensor(b!) special_out) -> ()",
    # out[i] = sum_c weight[i, c] * table[index[i, c]]: table [M, D], index [N, 4] int32,
    # weight [N, 4] fp32 -> [N, D] in the table's dtype; `order` (int32 [N]) only sets the
    # order the rows are computed in.  Zero weights skip their gather; an out-of-range index
    # with a non-zero weight yields a NaN row (the kernel never reads outside the table).
    "top4_project(Tensor table, Tensor index, Tensor weight) -> Tensor",
    "top4_project_into(Tensor table, Tensor index, Tensor weight, Tensor(a!) out) -> ()",
    "top4_project_ordered_into(Tensor table, Tensor index, Tensor weight, Tensor order, Tensor(a!) out) -> ()",
    # Segmented weighted pooling of x ([N, C] or [H, N, 64] view) into out; the LayerNorm
    # normalises every gathered row per 64-channel head first.  The multi form pools 1-3
    # channel ranges of one [N, W] row table in one launch (outputs of x's dtype, one eps).
    "compact_into(Tensor x, Tensor(a!) out, Tensor? base_rows, Tensor offsets, SymInt segs_per_row, "
    "Tensor? items, SymInt item_shift, Tensor? item_rows, Tensor? weights, Tensor? normalizer, "
    "Tensor? ln_weight, Tensor? ln_bias, float ln_eps) -> ()",
    "compact_multi_into(Tensor x, SymInt[] x_offsets, Tensor(a!)[] outs, Tensor?[] ln_weights, "
    "Tensor?[] ln_biases, float[] ln_eps, Tensor? base_rows, Tensor offsets, SymInt segs_per_row, "
    "Tensor? items, SymInt item_shift, Tensor? item_rows, Tensor? weights, Tensor? normalizer) -> ()",
    # [q, k, v] head-major [S, H, tokens_out, 64]; an unwanted one is an empty tensor.
    "qkv_epilogue(Tensor qkv, SymInt heads, SymInt tokens_in, SymInt tokens_out, Tensor? rows, "
    "Tensor? q_weight, Tensor? q_bias, Tensor? k_weight, Tensor? k_bias, float eps, Tensor? rope_sin, "
    "Tensor? rope_cos, SymInt rope_prefix, bool[] want, ScalarType out_dtype) -> Tensor[]",
    # [x + gamma * branch, LN in norm_dtype, LN in fp32, LN / max(||LN||, unit_eps)]; outputs not
    # asked for (no branch or write_sum false, no norm / norm_dtype, norm_f32 false,
    # unit_eps < 0) are empty tensors.
    "residual_layer_norm(Tensor x, Tensor? branch, Tensor? gamma, Tensor? ln_weight, Tensor? ln_bias, "
    "float eps, bool has_norm, bool write_sum, ScalarType? norm_dtype, bool norm_f32, float unit_eps) -> Tensor[]",
    # [x + gamma * restore(table), LN of that in norm_dtype] with restore = the top-4 projection
    # of `table` by (index, weight) -- or, without weight, the one-hot gather table[index] (zero
    # rows for index < 0) -- never written to memory.
    "restore_residual_layer_norm(Tensor x, Tensor table, Tensor index, Tensor? weight, Tensor? gamma, "
    "Tensor? ln_weight, Tensor? ln_bias, float eps, ScalarType norm_dtype) -> Tensor[]",
    "mlp_tail(Tensor x, Tensor h, Tensor fc1_weight, Tensor? fc1_bias, Tensor fc2_weight, Tensor? fc2_bias, "
    "Tensor? gamma) -> Tensor",
    "dense_block(Tensor x, Tensor?[] norms, float[] eps, Tensor?[] linears, Tensor?[] gammas, int heads, "
    "Tensor? rope_sin, Tensor? rope_cos, ScalarType dtype) -> Tensor",
    "merged_block(Tensor x, Tensor? h, Tensor? qkv, Tensor offsets, Tensor order, Tensor counts, "
    "Tensor? contribution, Tensor inverse, Tensor? log_mass, Tensor?[] norms, float[] eps, Tensor?[] linears, "
    "Tensor?[] gammas, int heads, ScalarType dtype) -> Tensor",
    "similarity_topk(Tensor src, Tensor dictionary, int topk, Tensor? src_rows, Tensor? n_src_device, int n_src, "
    "int n0, int off1, int n_dict, Tensor? index_map, Tensor(a!)? values, Tensor(b!) index, "
    "Tensor(c!)? scores) -> ()",
    "fastvggt_match(Tensor tokens, Tensor sources, Tensor destinations, bool prenormalized) -> (Tensor, Tensor)",
    "normalize_rows(Tensor x, Tensor? rows, float eps, ScalarType out_dtype) -> Tensor",
    "rope_table(Tensor(a!) sin, Tensor(b!) cos, int h, int w, float base) -> ()",
    "csr_build(Tensor keys, int n_buckets) -> (Tensor, Tensor)",
    "corner_csr(Tensor parent, int n_dest) -> (Tensor, Tensor)",
    "segment_mass(Tensor offsets, int segs_per_row, Tensor order, Tensor? weights, int rows, float start, "
    "bool want_log) -> (Tensor, Tensor)",
    "fastvggt_assemble(Tensor best, Tensor target, Tensor sources, Tensor destinations, int total, "
    "int removed) -> (Tensor, Tensor, Tensor)",
    "fastvggt_plan(Tensor best, Tensor target, Tensor sources, Tensor destinations, int total, "
    "int removed) -> Tensor[]",
)

_library = torch.library.Library("vgo", "DEF")
for _schema in _SCHEMAS:
    _library.define(_schema, tags=(torch.Tag.pt2_compliant_tag,))
_lib.load_ops_or_stubs([_schema.split("(")[0] for _schema in _SCHEMAS])


def _fake(name):
    return torch.library.register_fake("vgo::" + name, lib=_library)


@_fake("mass_bias_attention")
def _(q, k, v, log_key_mass):
    return torch.empty(q.shape, device=q.device, dtype=q.dtype)


@_fake("attention_into")
def _(q, k, v, bias, out, split):
    return None


@_fake("attention_pair_into")
def _(q, k, v, bias, out, special_q, special_k, special_v, special_bias, special_out):
    return None


@_fake("top4_project")
def _(table, index, weight):
    return table.new_empty((index.shape[0], table.shape[1]))


@_fake("top4_project_into")
def _(table, index, weight, out):
    return None


@_fake("top4_project_ordered_into")
def _(table, index, weight, order, out):
    return None


@_fake("compact_into")
def _(x, out, base_rows, offsets, segs_per_row, items, item_shift, item_rows, weights,
      normalizer, ln_weight, ln_bias, ln_eps):
    return None


@_fake("compact_multi_into")
def _(x, x_offsets, outs, ln_weights, ln_biases, ln_eps, base_rows, offsets, segs_per_row, items,
      item_shift, item_rows, weights, normalizer):
    return None


@_fake("qkv_epilogue")
def _(qkv, heads, tokens_in, tokens_out, rows, q_weight, q_bias, k_weight, k_bias, eps, rope_sin,
      rope_cos, rope_prefix, want, out_dtype):
    n_out = qkv.shape[0] if rows is None else rows.numel()
    shape = (n_out // tokens_out, heads, tokens_out, 64)
    return [qkv.new_empty(shape if w else (0,), dtype=out_dtype) for w in want]


@_fake("residual_layer_norm")
def _(x, branch, gamma, ln_weight, ln_bias, eps, has_norm, write_sum, norm_dtype, norm_f32, unit_eps):
    empty = x.new_empty((0,))
    total = x.new_empty(x.shape) if write_sum and branch is not None else empty
    normed = x.new_empty(x.shape, dtype=norm_dtype) if has_norm and norm_dtype is not None else empty
    normed32 = x.new_empty(x.shape) if has_norm and norm_f32 else empty
    unit = x.new_empty(x.shape, dtype=norm_dtype) if unit_eps >= 0 and norm_dtype is not None else empty
    return [total, normed, normed32, unit]


@_fake("restore_residual_layer_norm")
def _(x, table, index, weight, gamma, ln_weight, ln_bias, eps, norm_dtype):
    return [x.new_empty(x.shape), x.new_empty(x.shape, dtype=norm_dtype)]


@_fake("normalize_rows")
def _(x, rows, eps, out_dtype):
    n = x.numel() // x.shape[-1] if rows is None else rows.numel()
    return x.new_empty((n, x.shape[-1]), dtype=out_dtype)


@_fake("similarity_topk")
def _(src, dictionary, topk, src_rows, n_src_device, n_src, n0, off1, n_dict, index_map, values, index, scores):
    return None


@_fake("fastvggt_match")
def _(tokens, sources, destinations, prenormalized):
    shape = (tokens.shape[0], sources.numel())
    return tokens.new_empty(shape, dtype=torch.float32), tokens.new_empty(shape, dtype=torch.int32)


@_fake("fastvggt_assemble")
def _(best, target, sources, destinations, total, removed):
    batch = best.shape[0]
    return (sources.new_empty((batch, total - removed)), sources.new_empty((batch, total)),
            sources.new_empty(best.shape, dtype=torch.uint8))


@_fake("csr_build")
def _(keys, n_buckets):
    return (keys.new_empty((keys.numel(),), dtype=torch.int32),
            keys.new_empty((n_buckets + 1,), dtype=torch.int32))


@_fake("corner_csr")
def _(parent, n_dest):
    return (parent.new_empty((parent.numel(),), dtype=torch.int32),
            parent.new_empty((n_dest * parent.shape[-1] + 1,), dtype=torch.int32))


@_fake("segment_mass")
def _(offsets, segs_per_row, order, weights, rows, start, want_log):
    return (offsets.new_empty((rows,), dtype=torch.float32),
            offsets.new_empty((rows if want_log else 0,), dtype=torch.float32))


@_fake("fastvggt_plan")
def _(best, target, sources, destinations, total, removed):
    kept, n_src = total - removed, sources.numel()
    i32, f32 = dict(dtype=torch.int32), dict(dtype=torch.float32)
    return [sources.new_empty((1, kept)), sources.new_empty((1, total)),
            sources.new_empty((1, n_src), dtype=torch.uint8), sources.new_empty((total,), **i32),
            sources.new_empty((total,), **i32), sources.new_empty((kept + 1,), **i32),
            sources.new_empty((kept,), **f32), sources.new_empty((kept,), **f32)]
