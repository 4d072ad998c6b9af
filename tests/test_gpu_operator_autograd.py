"""What autograd sees of the operators: the path's refuse a backward and end tangents, the planners' leave no trace."""
from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

from tests.conftest import import_package

pytestmark = pytest.mark.gpu

N, K, C = 90, 41, 128


def _plan(vgo, device):
    return vgo.TokenPlan(torch.arange(K, device=device)[None], (torch.arange(N, device=device) % K)[None], N)


def _parents(device, requires_grad=False):
    g = torch.Generator(device=device).manual_seed(3)
    parent = torch.randint(0, K, (1, N - K, 4), device=device, generator=g)
    weight = torch.rand(1, N - K, 4, device=device, generator=g)
    return parent, weight.requires_grad_(requires_grad)


def test_plans_of_tensors_that_require_grad(vgo, device):
    kern = import_package("_kernels")
    parent, weight = _parents(device, requires_grad=True)
    mass = vgo.deterministic_weighted_normalizer(parent, weight, K)
    plan = vgo.WeightedBilinearTokenPlan(
        keep=torch.arange(K, device=device)[None], source_original=torch.arange(K, N, device=device)[None],
        source_parent_compact=parent, source_pool_weights=weight, source_restore_weights=weight, original_tokens=N,
        normalizer=mass)
    rows = kern.normalize_rows(torch.randn(20, C, device=device, requires_grad=True), None, 1e-12)
    for t in (mass, *plan.plan_mass(), rows):
        assert not t.requires_grad
    mass.cpu().numpy()
    assert torch.equal(mass, vgo.deterministic_weighted_normalizer(parent, weight.detach(), K))


def test_planners_refuse_function_transforms(vgo, device):
    """Where they would drop a derivative without a word."""
    kern = import_package("_kernels")
    parent, weight = _parents(device)
    rows = torch.randn(20, C, device=device)
    for call, t in ((lambda t: vgo.deterministic_weighted_normalizer(parent, t, K).sum(), weight),
                    (lambda t: kern.normalize_rows(t, None, 1e-12).float().sum(), rows),
                    (lambda t: _plan(vgo, device).compact(t).sum(), torch.randn(1, N, C, device=device)),
                    (lambda t: kern.similarity_topk(t.bfloat16(), rows.bfloat16(), 4)[0].sum(), rows)):
        for transform in (lambda f, t: torch.func.grad(f)(t), lambda f, t: torch.func.jvp(f, (t,), (t,)),
                          lambda f, t: torch.func.vmap(f)(t[None])):
            with pytest.raises(RuntimeError):
                transform(call, t)


def test_path_outputs_refuse_a_backward(vgo, device):
    index, w = torch.zeros(5, 4, dtype=torch.int32, device=device), torch.rand(5, 4, device=device)
    out = vgo.top4_project(torch.randn(8, 16, device=device, requires_grad=True), index, w)
    assert out.requires_grad
    with pytest.raises(RuntimeError, match="top4_project"):
        out.sum().backward()
    with torch.no_grad():
        assert not vgo.top4_project(torch.randn(8, 16, device=device, requires_grad=True), index, w).requires_grad


@pytest.mark.parametrize("grad", [True, False])
def test_tangents_end_at_the_path(vgo, device, grad):
    """As with inputs that require no grad: the values are those of the plain call, without a tangent."""
    torch.manual_seed(4)
    block = vgo.SelfAttentionBlock(C, 2, use_qk_norm=True, init_values=0.5).eval().to(device)
    table, x = torch.randn(20, C, device=device), torch.randn(1, N, C, device=device)
    index = torch.randint(0, 20, (30, 4), dtype=torch.int32, device=device)
    w, q, mass = torch.rand(30, 4, device=device), torch.randn(1, 2, 50, 64, device=device), torch.randn(50, device=device)
    parent, weight = _parents(device)
    calls = [(lambda t: vgo.mass_bias_attention(t, q, q, mass), q), (lambda t: vgo.top4_project(t, index, w), table),
             (lambda t: _plan(vgo, device).compact(t), x), (lambda t: _plan(vgo, device).restore(t[:, :K]), x),
             (lambda t: vgo.deterministic_weighted_normalizer(parent, t, K), weight)]
    if not grad:  # the blocks' own parameters require grad
        calls += [(block, x), (lambda t: block.forward_compacted(t, _plan(vgo, device)), x)]
    with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16):
        for call, t in calls:
            expect = call(t)
            with forward_ad.dual_level():
                got = call(forward_ad.make_dual(t, torch.ones_like(t)))
                assert forward_ad.unpack_dual(got).tangent is None
            assert torch.equal(got, expect)
    with forward_ad.dual_level(), pytest.raises(NotImplementedError):
        vgo.top4_project(forward_ad.make_dual(table, table).requires_grad_(), index, w)


def test_outputs_written_in_place(vgo, device):
    """Any tensor may take the result; its version counts the write."""
    table, index = torch.randn(20, C, device=device), torch.randint(0, 20, (30, 4), dtype=torch.int32, device=device)
    w = torch.rand(30, 4, device=device)
    expect = vgo.top4_project(table, index, w)
    leaf = torch.zeros(30, C, device=device, requires_grad=True)
    plain = torch.zeros(30, C, device=device)
    with torch.inference_mode():
        inference = torch.zeros(30, C, device=device)
    for out in (leaf, plain, inference):
        before = None if out.is_inference() else out._version
        vgo.top4_project(table, index, w, out=out)
        assert torch.equal(out, expect) and out.grad_fn is None
        assert before is None or out._version > before


def test_vmap_runs_one_call_per_element(vgo, device):
    """Operators with new tensors as results run under vmap; those that write arguments, planners and blocks refuse."""
    g = torch.Generator(device=device).manual_seed(8)
    q, k, v = (torch.randn(3, 1, 2, 50, 64, device=device, generator=g) for _ in range(3))
    mass, table = torch.randn(50, device=device, generator=g), torch.randn(3, 20, C, device=device, generator=g)
    index = torch.randint(0, 20, (30, 4), dtype=torch.int32, device=device, generator=g)
    w = torch.rand(30, 4, device=device, generator=g)
    got = torch.func.vmap(lambda a, b, c: vgo.mass_bias_attention(a, b, c, mass))(q, k, v)
    assert torch.equal(got, torch.stack([vgo.mass_bias_attention(*t, mass) for t in zip(q, k, v)]))
    got = torch.func.vmap(lambda t: vgo.top4_project(t, index, w), in_dims=0, out_dims=1)(table)
    assert torch.equal(got, torch.stack([vgo.top4_project(t, index, w) for t in table], dim=1))
    none = [None] * 8
    for refused in (lambda t: vgo.top4_project(t, index, w, out=torch.empty(30, C, device=device)),
                    lambda t: torch.ops.vgo.residual_layer_norm(t, None, None, None, None, 1e-5, True, True,
                                                                torch.bfloat16, False, -1.0)[1],
                    lambda t: torch.ops.vgo.normalize_rows(t, None, 1e-12, torch.bfloat16),
                    lambda t: torch.ops.vgo.dense_block(t[None], none, [1e-5] * 3, none, none[:2], 2, None, None,
                                                        torch.bfloat16)):
        with pytest.raises(RuntimeError):
            torch.func.vmap(refused)(table)
