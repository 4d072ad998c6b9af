"""A FastVGGT plan from one launch against the launches it stands for, bit for bit."""
from __future__ import annotations

import pytest
import torch

from tests.conftest import import_package

pytestmark = pytest.mark.gpu


def _case(seed, ns, nd, rest, device, scores):
    """best, target, sources, destinations over ns + nd + rest tokens in a random interleaving."""
    g = torch.Generator().manual_seed(seed)
    total = ns + nd + rest
    ids = torch.randperm(total, generator=g)
    sources, destinations = ids[:ns].sort().values, ids[ns:ns + nd].sort().values
    target = torch.randint(0, nd, (1, ns), generator=g, dtype=torch.int32)
    if scores == "bf16":
        best = (torch.rand(1, ns, generator=g) * 2 - 1).bfloat16().float()
    elif scores == "fp32":
        best = torch.randn(1, ns, generator=g)
    elif scores == "tied":  # every key equal, every token onto one destination
        best = torch.full((1, ns), -0.5)
        target.fill_(nd // 2)
    else:
        best = torch.tensor([0.0, -0.0, float("nan"), -float("nan"), float("inf"), -float("inf"), 1e-40, -1.0])[
            torch.randint(0, 8, (1, ns), generator=g)]
        target[0, ::3] = 0
    return total, best.to(device), target.to(device), sources.to(device), destinations.to(device)


@pytest.mark.parametrize("scores", ["bf16", "fp32", "tied", "special"])
@pytest.mark.parametrize("ns,nd,rest", [(1, 1, 0), (63, 7, 2), (1024, 300, 5), (1025, 128, 900), (3000, 1000, 96),
                                        (3000, 1000, 97), (9000, 2500, 788)])
def test_one_launch_equals_the_launches(vgo, device, scores, ns, nd, rest):
    kern, lib = import_package("_kernels"), import_package("_lib").load()
    total, best, target, sources, destinations = _case(ns + nd, ns, nd, rest, device, scores)
    for removed in sorted({1, (ns + 1) // 2, ns}):
        assert lib.vgo_fastvggt_plan_fits(ns, total, removed)
        print(f"[plan] {scores} ns={ns} nd={nd} removed={removed}", flush=True)
        got = torch.ops.vgo.fastvggt_plan(best, target, sources, destinations, total, removed)
        keep, inverse, flags = torch.ops.vgo.fastvggt_assemble(best, target, sources, destinations, total, removed)
        order, offsets = kern.csr_build(inverse[0], total - removed)
        mass, log_mass = kern.segment_mass(offsets, 1, order, None, total - removed, 0.0)
        want = (keep, inverse, flags, inverse[0].int(), order, offsets, mass, log_mass)
        names = ("keep", "inverse", "flags", "inverse32", "order", "offsets", "mass", "log_mass")
        for name, a, b in zip(names, got, want):
            assert torch.equal(a, b), name


def test_plans_that_do_not_fit_take_the_launches(vgo, device):
    lib = import_package("_lib").load()
    assert lib.vgo_fastvggt_plan_fits(9000, 12288, 6000) and not lib.vgo_fastvggt_plan_fits(9000, 12289, 6000)
    total, best, target, sources, destinations = _case(1, 9000, 3000, 289, device, "bf16")
    with pytest.raises(RuntimeError, match="too many tokens"):
        torch.ops.vgo.fastvggt_plan(best, target, sources, destinations, total, 6000)


@pytest.mark.parametrize("mode", ["no_grad", "inference"])
@pytest.mark.parametrize("side", [8, 80])  # 195 and 19,203 tokens: the one launch, and the launches
def test_a_plan_changed_before_its_first_use_pools_as_changed(vgo, device, side, mode):
    """A mask, an inverse or its contents set on a built plan count, as on a plan constructed with them."""
    frames, special = 3, 1
    per_frame = special + side * side
    g = torch.Generator(device=device).manual_seed(side)
    x = torch.randn(1, frames * per_frame, 64, device=device, generator=g)

    def build():
        return vgo.build_fastvggt_plan(x, frames=frames, tokens_per_frame=per_frame, patch_token_start=special,
                                       patch_hw=(side, side), merge_ratio=0.5, protect_ratio=0.0)

    with torch.inference_mode() if mode == "inference" else torch.no_grad():
        plain = build()
        total, kept = plain.original_tokens, plain.kept_tokens
        print(f"[changed plan] {total} tokens, {kept} kept, {mode}", flush=True)
        counts = torch.bincount(plain.inverse[0].cpu(), minlength=kept)
        assert torch.equal(plain.cluster_counts().cpu(), counts.float())
        # Every cluster keeps its representative, so that no masked count is zero.
        mask = torch.rand(1, total, device=device, generator=g) < 0.5
        mask[0, plain.keep[0]] = True
        other = plain.inverse.flip(1)
        expect = vgo.TokenPlan(plain.keep, plain.inverse.clone(), total, pool_mask=mask)
        flipped = vgo.TokenPlan(plain.keep, other.clone(), total)

        masked = build()
        masked.pool_mask = mask
        assert torch.equal(masked.cluster_counts(), expect.cluster_counts())
        assert torch.equal(masked.compact(x), expect.compact(x)) and not torch.equal(masked.compact(x), plain.compact(x))
        replaced = build()
        replaced.inverse = other
        written = build()
        written.inverse.copy_(other)
        for plan in (replaced, written):
            assert torch.equal(plan._inverse32(0), other[0].int())
            assert torch.equal(plan.cluster_counts(), flipped.cluster_counts())
            assert torch.equal(plan.compact(x), flipped.compact(x))
