"""The key-split attention kernel (few tasks) and its border with the register-staged one.

Reference: the oracle's softmax(q k^T / 8 + log m) v on the rounded inputs; tolerance: the
repository's 2e-2 for bf16/f16 (probabilities are rounded to the type before P V).
"""
from __future__ import annotations

import pytest
import torch

from oracle import attention as oracle
from tests._tol import assert_close

pytestmark = pytest.mark.gpu


def _inputs(seed, b, h, nq, nk, dtype, std):
    g = torch.Generator().manual_seed(seed)
    q, k = ((torch.randn(b, h, n, 64, generator=g) * std).to(dtype) for n in (nq, nk))
    v = torch.randn(b, h, nk, 64, generator=g).to(dtype)
    return q, k, v, torch.randint(1, 9, (nk,), generator=g).float().log()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nq,nk", [(1, 1), (31, 64), (32, 65), (33, 256), (64, 257), (100, 320), (5, 2559)])
def test_key_split_edges(vgo, device, dtype, nq, nk):
    """Tiles that do not divide over the four waves, waves without a tile, ragged queries and
    keys; whole leading tiles of mass 0; heavy late keys, which move the reference maximum of
    some waves only; token-major views."""
    mba = __import__("importlib").import_module("4d_ttt_merging_amd.mass_bias_attention")
    for std in (0.125, 2.0):
        q, k, v, bias = _inputs(nq * 13 + nk, 2, 3, nq, nk, dtype, std)
        if nk > 100:
            bias[:70] = -float("inf")
            bias[nk - 20:] += 12.0
        qd, kd, vd = (t.transpose(1, 2).contiguous().to(device).transpose(1, 2) for t in (q, k, v))
        out = torch.full((2, nq, 3, 64), float("nan"), device=device, dtype=dtype)
        mba._attention_into(qd, kd, vd, bias.to(dtype).to(device), out.permute(0, 2, 1, 3), split=False)
        ref = oracle.mass_bias_attention(q, k, v, bias)
        assert_close(out.permute(0, 2, 1, 3).cpu(), ref, dtype, what=f"{dtype} {nq}x{nk} std {std}")


@pytest.mark.parametrize("heads", [3, 64])
def test_both_kernels_without_a_workspace(vgo, device, heads):
    """385 queries: 39 key-split work-groups at 3 heads; 832 at 64 heads, more than 768, so
    the register-staged kernel."""
    mba = __import__("importlib").import_module("4d_ttt_merging_amd.mass_bias_attention")
    q, k, v, bias = _inputs(heads, 1, heads, 385, 130, torch.bfloat16, 1.0)
    out = torch.empty(q.shape, device=device, dtype=q.dtype)
    mba._attention_into(q.to(device), k.to(device), v.to(device), bias.bfloat16().to(device), out, split=False)
    assert_close(out.cpu(), oracle.mass_bias_attention(q, k, v, bias), torch.bfloat16, what=f"{heads} heads")
