"""q, k and v of a four-parent plan pooled by one launch against one output at a time."""
from __future__ import annotations

import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


def _plan(vgo, device, total, removed, **kw):
    g = torch.Generator().manual_seed(total + removed)
    source = torch.randperm(total, generator=g)[:removed].sort().values
    mask = torch.ones(total, dtype=torch.bool)
    mask[source] = False
    keep = mask.nonzero().flatten()
    parent = torch.randint(0, keep.numel(), (removed, 4), generator=g)
    weight = torch.rand(removed, 4, generator=g)
    mass = torch.ones(keep.numel()).index_add_(0, parent.flatten(), weight.flatten())
    keep, source, parent, weight, mass = (t.to(device) for t in (keep, source, parent, weight, mass))
    return vgo.WeightedBilinearTokenPlan(
        keep=keep[None], source_original=source[None], source_parent_compact=parent[None],
        source_pool_weights=weight[None], source_restore_weights=weight[None], original_tokens=total,
        normalizer=mass.view(1, -1, 1), key_log_mass=mass.log().view(1, -1), **kw)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("total,removed", [(9, 1), (70, 69), (261, 100)])
@pytest.mark.parametrize("kw,together", [(dict(), True), (dict(preserve_queries=True), True),
                                         (dict(preserve_queries=True, preserve_destination_keys=True), False),
                                         (dict(pool_source_content=False), False)])
def test_layer_equals_one_output_at_a_time(vgo, device, monkeypatch, dtype, total, removed, kw, together):
    torch.manual_seed(total)
    plan = _plan(vgo, device, total, removed, **kw)
    assert plan.pools_qkv_together() == together
    layers = importlib.import_module("4d_ttt_merging_amd.layers")
    rows = torch.randn(total * 384 + 1, device=device).to(dtype)
    for norm, offset in ((True, 0), (False, 0), (False, 1)):
        if offset and (kw.get("preserve_queries") or dtype != torch.float32):
            continue  # rows off the 16-byte grid: only the launch per output, without a norm, takes them
        layer = vgo.SelfAttention(128, num_heads=2, qkv_bias=True, use_qk_norm=norm, device=device).eval().to(device)
        for p in layer.parameters():
            torch.nn.init.normal_(p, std=0.2)
        qkv = rows[offset:offset + total * 384].view(1, total, 384)
        assert layers._vector_rows(qkv[0]) == (offset == 0)
        with torch.no_grad():
            out = layer.compute_attention(qkv, token_plan=plan)
            with monkeypatch.context() as m:
                m.setattr(type(plan), "pools_qkv_together", lambda self: False)
                assert torch.equal(out, layer.compute_attention(qkv, token_plan=plan))
