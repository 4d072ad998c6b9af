"""fp32 attention on the matrix cores: tile edges, cut tasks, and both row layouts.

The reference is softmax(q k^T / 8 + bias) v in float64.  Bound: products and
sums are fp32 (2^-24 each); a 32-key chunk's sums and the chain of nk / 32 chunk
sums each grow like a random walk, and |logits| <= 8 adds 8 * 2^-24 to an
exponent: below 1e-5 of max(|out|, rms) at these sizes (the repository's fp32
tolerance).
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from tests._tol import assert_close

pytestmark = pytest.mark.gpu


def _reference(q, k, v, bias):
    s = q.double() @ k.double().transpose(-1, -2) / 8
    if bias is not None:
        s = s + bias.double()
    return torch.softmax(s, -1) @ v.double()


def _operands(seed, batch, heads, nq, nk, layout, device):
    """q, k, v, out as [batch, heads, n, 64] views: head-major, token-major, or rows that
    start at odd 4-byte addresses (no 16-byte access possible)."""
    g = torch.Generator().manual_seed(seed)
    views = []
    for n in (nq, nk, nk, nq):
        x = torch.randn(batch, heads, n, 64, generator=g)
        if layout == "head":
            t = x.to(device)
        elif layout == "token":
            t = x.transpose(1, 2).contiguous().to(device).transpose(1, 2)
        else:
            t = torch.zeros(batch, heads, n, 67).to(device)[..., 1:65]
            t.copy_(x)
        views.append(t)
    return views


@pytest.mark.parametrize("layout", ["head", "token", "odd"])
@pytest.mark.parametrize("nq,nk", [(1, 1), (31, 33), (64, 64), (65, 63), (256, 65), (257, 128), (321, 1000)])
def test_tile_edges(vgo, device, layout, nq, nk):
    mba = __import__("importlib").import_module("4d_ttt_merging_amd.mass_bias_attention")
    q, k, v, out = _operands(nq * 7 + nk, 2, 3, nq, nk, layout, device)
    bias = torch.randint(1, 9, (nk,), generator=torch.Generator().manual_seed(nk)).float().log()
    if nk > 40:
        bias[:35] = -float("inf")  # a whole leading 32-key chunk of mass 0
    for b in (bias, None):
        ref = _reference(q.cpu(), k.cpu(), v.cpu(), b)
        for split in (None, False):  # cut between work-groups; one task per work-group
            out.fill_(float("nan"))
            mba._attention_into(q, k, v, None if b is None else b.to(device), out, split=split)
            assert_close(out.cpu(), ref, torch.float32, what=f"{layout} split={split} bias={b is not None}")


@pytest.mark.parametrize("split", [None, False])
@pytest.mark.parametrize("batch", [16_400, 70_000, (1 << 20) + 3])
def test_many_small_problems(vgo, device, batch, split):
    """Tasks past those that are cut, past the merge's grid, and past a grid of one task per work-group.

    With one key the result is its value, in whatever order it is computed."""
    mba = __import__("importlib").import_module("4d_ttt_merging_amd.mass_bias_attention")
    heads = 2 if batch < 20_000 else 16
    g = torch.Generator(device=device).manual_seed(batch)
    q = torch.randn(batch, heads, 1, 64, device=device, generator=g)
    v = torch.randn(batch, heads, 1, 64, device=device, generator=g)
    out = torch.full_like(v, float("nan"))
    mba._attention_into(q, q, v, None, out, split=split)
    assert torch.equal(out, v)
    if batch < 100_000:  # two key tiles each, shared by all batch elements
        k, v = (torch.randn(1, heads, 65, 64, device=device, generator=g).expand(batch, -1, -1, -1) for _ in range(2))
        mba._attention_into(q, k, v, None, out.fill_(float("nan")), split=split)
        for rows in (slice(0, 50), slice(batch // 2, batch // 2 + 50), slice(batch - 50, batch)):
            assert_close(out[rows].cpu(), _reference(*(t[rows].cpu() for t in (q, k, v)), None), torch.float32)
        assert torch.isfinite(out).all()


def test_split_workspace_is_checked(vgo, device):
    lib_mod = __import__("importlib").import_module("4d_ttt_merging_amd._lib")
    lib = lib_mod.load()
    q, k, v, out = _operands(3, 1, 2, 300, 500, "head", device)
    need = ctypes.c_size_t(0)
    lib_mod.check(lib.vgo_mass_bias_attn_f32_workspace(1, 2, 300, 500, ctypes.byref(need)))
    assert need.value > 0
    s = [lib_mod.strides3(t) for t in (q, k, v, out)]
    with pytest.raises(RuntimeError, match="workspace too small"):
        lib_mod.check(lib.vgo_mass_bias_attn_f32_fwd_ws(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), None, out.data_ptr(), 1, 2, 300, 500, 64, *s, None, 0,
            lib_mod.stream_of(q)))
