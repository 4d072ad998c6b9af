"""Typed wrappers over the merge-path entry points of `libvgo.so`.

The wrappers go through the torch.library operators of `ops.py`
(`torch.ops.vgo.*`, implemented in csrc/torch_ops.cpp), which check shapes and
dtypes, allocate outputs and workspaces with torch and launch on torch's
current stream; the restore map calls the C ABI directly.  No wrapper
synchronises the device.
"""
from __future__ import annotations

import torch

from . import _lib


def _c(ptr_or_tensor):
    if ptr_or_tensor is None:
        return None
    return ptr_or_tensor.data_ptr()


def normalize_rows(x: torch.Tensor, rows: torch.Tensor | None, eps: float,
                   out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """out[r] = x[rows[r]] / max(||x[rows[r]]||, eps) for a 2-D x (unit column stride)."""
    _lib.require_plain(x, rows)
    return torch.ops.vgo.normalize_rows(x, rows, float(eps), out_dtype)


def similarity_topk(src: torch.Tensor, dictionary: torch.Tensor, topk: int, *,
                    src_rows: torch.Tensor | None = None,
                    n_src_device: torch.Tensor | None = None, n_src: int | None = None,
                    dict_ranges: tuple[int, int, int] | None = None,
                    index_map: torch.Tensor | None = None, want_values: bool = True,
                    index_dtype: torch.dtype = torch.int64,
                    scores: torch.Tensor | None = None,
                    out: tuple[torch.Tensor, torch.Tensor] | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """Top-K bf16 cosine matches of every source row against a dictionary.

    dict_ranges = (n0, off1, n_dict): dictionary position j reads row j for
    j < n0 and row off1 + j - n0 otherwise (default: all rows).  Returns
    (values [n, K] fp32, indices [n, K]) with ties going to the lower position,
    written into `out` = (values, indices) when given (contiguous, those shapes).
    """
    _lib.load()
    _lib.require_gpu(src, dictionary, src_rows, n_src_device, index_map, scores)
    _lib.require_plain(src, dictionary, src_rows, n_src_device, index_map, scores)
    if src.dtype != torch.bfloat16 or dictionary.dtype != torch.bfloat16:
        raise ValueError("similarity_topk expects bf16 operands")
    if dict_ranges is None:
        dict_ranges = (dictionary.shape[0], 0, dictionary.shape[0])
    n0, off1, n_dict = dict_ranges
    if n_src is None:
        n_src = src.shape[0] if src_rows is None else src_rows.numel()
    if out is not None:
        values, index = out
        if index.dtype != index_dtype:
            raise ValueError("similarity_topk: `out` must be contiguous [n, K] fp32 values and indices")
    else:
        values = torch.empty((n_src, topk), device=src.device, dtype=torch.float32) if want_values else None
        index = torch.empty((n_src, topk), device=src.device, dtype=index_dtype)
    torch.ops.vgo.similarity_topk(src, dictionary, topk, src_rows, n_src_device, n_src, n0, off1, n_dict,
                                  index_map, values, index, scores)
    return values, index


def csr_build(keys: torch.Tensor, n_buckets: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Stable bucket order: (order [n] int32 item ids, offsets [n_buckets+1] int32)."""
    _lib.require_plain(keys)
    return torch.ops.vgo.csr_build(keys, n_buckets)


def corner_csr(parent: torch.Tensor, n_dest: int) -> tuple[torch.Tensor, torch.Tensor]:
    """csr_build of the (destination, corner) pairs: item p = i*S + c, key = parent*S + c of [M, S] parents."""
    _lib.require_plain(parent)
    return torch.ops.vgo.corner_csr(parent, n_dest)


def segment_mass(offsets: torch.Tensor, segs_per_row: int, order: torch.Tensor,
                 weights: torch.Tensor | None, rows: int, start: float,
                 want_log: bool = True) -> tuple[torch.Tensor, torch.Tensor | None]:
    """Sequential per-segment sums from `start` (fp32 [rows]) and, if asked, their logarithms."""
    _lib.require_plain(offsets, order, weights)
    mass, log_mass = torch.ops.vgo.segment_mass(offsets, segs_per_row, order, weights, rows, float(start),
                                                want_log)
    return mass, log_mass if want_log else None


def restore_map(total: int, *, device: torch.device, keep: torch.Tensor | None = None,
                source: torch.Tensor | None = None, parent: torch.Tensor | None = None,
                weight: torch.Tensor | None = None,
                inverse: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """Dense [total, 4] (int32 index, fp32 weight) rows consumed by top4_project."""
    lib = _lib.load()
    _lib.require_gpu(keep, source, parent, weight, inverse)
    n_keep = 0 if keep is None else keep.numel()
    n_source = 0 if source is None else source.numel()
    if inverse is not None and inverse.numel() < total:
        raise ValueError(f"restore_map: {inverse.numel()} inverse entries for {total} tokens")
    if n_source and (parent is None or weight is None or min(parent.numel(), weight.numel()) < 4 * n_source):
        raise ValueError("restore_map: four parents and weights per source")
    # With `inverse` the kernel writes every row; otherwise rows outside keep and
    # source stay zero (zero weights, as the reference's `new_zeros` output).
    if inverse is not None:
        index_out = torch.empty((total, 4), device=device, dtype=torch.int32)
        weight_out = torch.empty((total, 4), device=device, dtype=torch.float32)
    else:  # one fill for both
        index_out, weight_out = torch.zeros((2, total, 4), device=device, dtype=torch.int32).unbind()
        weight_out = weight_out.view(torch.float32)
    status = lib.vgo_restore_map(
        _c(keep), n_keep, _c(source), _c(parent), _c(weight), n_source, _c(inverse), total,
        index_out.data_ptr(), weight_out.data_ptr(), torch.cuda.current_stream(device).cuda_stream)
    _lib.check(status)
    return index_out, weight_out


# --------------------------------------------- operator-backed entry points ----
def compact_into(x: torch.Tensor, out: torch.Tensor, *, base_rows: torch.Tensor | None,
                 offsets: torch.Tensor, segs_per_row: int, items: torch.Tensor | None,
                 item_shift: int, item_rows: torch.Tensor | None, weights: torch.Tensor | None,
                 normalizer: torch.Tensor | None,
                 layer_norm: tuple[torch.Tensor, torch.Tensor, float] | None = None) -> torch.Tensor:
    """Segmented weighted pooling into `out` (torch.ops.vgo.compact_into): x/out are
    [N, C] or head-major [H, N, 64] views.

    `layer_norm` = (weight [64], bias [64], eps) normalises every gathered row per
    64-channel head first; `out` may be narrower than `x` (one final rounding)."""
    ln_w, ln_b, eps = layer_norm if layer_norm is not None else (None, None, 0.0)
    torch.ops.vgo.compact_into(x, out, base_rows, offsets, segs_per_row, items, item_shift, item_rows,
                               weights, normalizer, ln_w, ln_b, float(eps))
    return out


def compact_multi_into(x: torch.Tensor, outputs, *, base_rows: torch.Tensor | None,
                       offsets: torch.Tensor, segs_per_row: int, items: torch.Tensor | None,
                       item_shift: int, item_rows: torch.Tensor | None, weights: torch.Tensor | None,
                       normalizer: torch.Tensor | None) -> None:
    """1-3 outputs of one segment structure in one launch (torch.ops.vgo.compact_multi_into);
    `outputs` holds (channel offset, out, layer_norm or None) per output."""
    torch.ops.vgo.compact_multi_into(
        x, [int(off) for off, _, _ in outputs], [out for _, out, _ in outputs],
        [None if ln is None else ln[0] for _, _, ln in outputs],
        [None if ln is None else ln[1] for _, _, ln in outputs],
        [0.0 if ln is None else float(ln[2]) for _, _, ln in outputs],
        base_rows, offsets, segs_per_row, items, item_shift, item_rows, weights, normalizer)


def qkv_epilogue(qkv: torch.Tensor, heads: int, *, tokens_in: int, tokens_out: int | None = None,
                 rows: torch.Tensor | None = None, q_norm=None, k_norm=None, eps: float = 1e-5,
                 rope: tuple[torch.Tensor, torch.Tensor] | None = None, rope_prefix: int = 0,
                 want=(True, True, True), out_dtype: torch.dtype | None = None):
    """Split packed qkv rows [T, 3C] into head-major [S, H, tokens_out, 64] q/k/v
    (torch.ops.vgo.qkv_epilogue).

    q_norm / k_norm are (weight, bias) of the per-head LayerNorm(64); rope is
    (sin, cos) [positions, 64] applied to tokens at position >= rope_prefix of
    each tokens_in-long sequence.  Returns (q, k, v) with None for unwanted ones."""
    outs = torch.ops.vgo.qkv_epilogue(
        qkv, heads, tokens_in, tokens_out or tokens_in, rows,
        None if q_norm is None else q_norm[0], None if q_norm is None else q_norm[1],
        None if k_norm is None else k_norm[0], None if k_norm is None else k_norm[1], float(eps),
        None if rope is None else rope[0], None if rope is None else rope[1], rope_prefix,
        [bool(w) for w in want], out_dtype or qkv.dtype)
    return tuple(o if w else None for o, w in zip(outs, want))


def residual_layer_norm(x: torch.Tensor, branch: torch.Tensor | None = None,
                        gamma: torch.Tensor | None = None,
                        norm: tuple[torch.Tensor | None, torch.Tensor | None, float] | None = None, *,
                        write_sum: bool = True, norm_dtype: torch.dtype | None = torch.bfloat16,
                        norm_f32: bool = False, unit_eps: float | None = None):
    """One pass over fp32 rows [..., dim] (torch.ops.vgo.residual_layer_norm):
    s = x + gamma * branch, n = LayerNorm(s).

    `norm` = (weight, bias, eps) of the LayerNorm (affine tensors may be None).
    Returns (s, n, n_f32[, u]): s when `write_sum` (and a branch is given), n in
    `norm_dtype` and its fp32 copy when asked, else None in their places; with
    `unit_eps`, also u = n / max(||n||, unit_eps) in `norm_dtype` (the planners'
    F.normalize front end, equal bit for bit to normalize_rows of n_f32)."""
    w, b, eps = norm if norm is not None else (None, None, 0.0)
    outs = torch.ops.vgo.residual_layer_norm(
        x, branch, gamma, w, b, float(eps), norm is not None, write_sum, norm_dtype, norm_f32,
        -1.0 if unit_eps is None else float(unit_eps))
    total = outs[0] if write_sum and branch is not None else None
    normed = outs[1] if norm is not None and norm_dtype is not None else None
    normed32 = outs[2] if norm is not None and norm_f32 else None
    if unit_eps is not None:
        return total, normed, normed32, outs[3]
    return total, normed, normed32


def restore_residual_layer_norm(x: torch.Tensor, table: torch.Tensor, index: torch.Tensor,
                                weight: torch.Tensor | None, gamma: torch.Tensor | None,
                                norm: tuple[torch.Tensor | None, torch.Tensor | None, float], *,
                                norm_dtype: torch.dtype = torch.bfloat16):
    """One pass over fp32 rows x [N, dim] with the branch restored from `table` on the fly
    (torch.ops.vgo.restore_residual_layer_norm): branch = top4_project(table, index, weight)
    (same rounding), s = x + gamma * branch, n = LayerNorm(s) in `norm_dtype`.  With weight
    None, index is a one-hot int32 [N] map (a token plan's inverse): branch = table[index]
    (zero rows for index < 0).  Returns (s, n)."""
    w, b, eps = norm
    total, normed = torch.ops.vgo.restore_residual_layer_norm(x, table, index, weight, gamma, w, b,
                                                              float(eps), norm_dtype)
    return total, normed
