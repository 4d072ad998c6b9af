"""The RoPE tables from one launch: the values of torch's operators, and close to 64 bits."""
from __future__ import annotations

import math

import pytest
import torch

from tests.conftest import import_package

pytestmark = pytest.mark.gpu


def _exact(h, w, dim, base):
    periods = base ** (2 * torch.arange(dim // 4, dtype=torch.float64) / (dim // 2))
    y, x = torch.arange(0.5, h, dtype=torch.float64) / max(h, w), torch.arange(0.5, w, dtype=torch.float64) / max(h, w)
    coords = 2 * torch.stack(torch.meshgrid(y, x, indexing="ij"), dim=-1).flatten(0, 1) - 1
    angles = (2 * math.pi * coords[:, :, None] / periods).flatten(1, 2).tile(2)
    return angles.sin(), angles.cos()


@pytest.mark.parametrize("h,w,dim,base", [(1, 1, 64, 100.0), (1, 37, 64, 100.0), (37, 1, 4, 100.0), (27, 35, 64, 100.0),
                                          (32, 32, 64, 100.0), (13, 8, 12, 10000), (200, 300, 128, 2.5)])
def test_tables(vgo, device, h, w, dim, base):
    layers = import_package("layers")
    print(f"[rope] {h} x {w} x {dim}", flush=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        sin, cos = layers.rope_sincos(h, w, dim, base, device=device)
        with _TorchOnly():
            torch_sin, torch_cos = layers.rope_sincos(h, w, dim, base, device=device)
    assert sin.shape == (h * w, dim) and sin.dtype == torch.float32 and sin.is_contiguous() and cos.is_contiguous()
    # An angle of up to 2 pi carries the roundings of five operations and of the power (2 ulp).
    bound = 2 * math.pi * 8 * 2.0 ** -24 + 2.0 ** -23
    for ours, theirs, exact in zip((sin, cos), (torch_sin, torch_cos), _exact(h, w, dim, base)):
        assert torch.equal(ours, theirs)
        assert float((ours.cpu().double() - exact).abs().max()) <= bound


class _TorchOnly(torch.overrides.TorchFunctionMode):
    """Any function mode: rope_sincos then takes torch's operators."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_transforms_and_devices_take_torch_operators(vgo, device):
    layers = import_package("layers")
    assert layers.rope_sincos(3, 4, 8)[0].device.type == "cpu"
    x = torch.randn(5, 12, 8, device=device)
    out = torch.func.vmap(lambda v: v * layers.rope_sincos(3, 4, 8, device=device)[0])(x)
    assert torch.equal(out, x * layers.rope_sincos(3, 4, 8, device=device)[0])


def test_sizes_past_the_kernel_take_torch_operators(vgo, device):
    """The kernel's limits: 2^20 rows or columns of patches, 2^31 values."""
    layers = import_package("layers")
    for h, w, dim in ((1 << 20, 1, 4), (1, 1 << 20, 4), (1 << 10, 1 << 11, 1024)):
        assert not layers._one_launch_rope(h, w, dim, 100.0, device)
        assert layers._one_launch_rope(h - (h > 1), w - (w > 1), dim, 100.0, device)
    sin, cos = layers.rope_sincos(1 << 20, 1, 4, device=device)
    with _TorchOnly():
        expect = layers.rope_sincos(1 << 20, 1, 4, device=device)
    assert torch.equal(sin, expect[0]) and torch.equal(cos, expect[1])


def test_tables_are_tensors_of_their_own(vgo, device):
    """Each may be written in place, under autograd too, without a trace in the other."""
    layers = import_package("layers")
    sin, cos = layers.rope_sincos(3, 4, 8, device=device)
    expect, version = sin.clone(), cos._version
    assert not sin._is_view() and sin.untyped_storage().data_ptr() != cos.untyped_storage().data_ptr()
    scale = torch.full((8,), 2.0, device=device, requires_grad=True)
    sin.mul_(scale)
    sin.sum().backward()
    assert torch.equal(sin.detach(), 2 * expect) and torch.equal(scale.grad, expect.sum(0)) and cos._version == version
