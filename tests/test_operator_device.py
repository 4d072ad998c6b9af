"""The operators launch on their tensors' device, whichever device is current."""
from __future__ import annotations

import re

import pytest
import torch

from tests.conftest import PACKAGE, ROOT, import_package


def test_every_operator_sets_its_device():
    """Each registered implementation goes through the device guard, and each schema has one."""
    source = (ROOT / PACKAGE / "csrc" / "torch_ops.cpp").read_text()
    block = re.search(r"void register_cuda\(torch::Library& m\) \{(.*?)\n\}", source, re.S).group(1)
    implementations = re.findall(r'm\.impl\("(\w+)",\s*(.*?)\);', block)
    assert {f"on_device<{name}>" for name, _ in implementations} == {how for _, how in implementations}
    schemas = import_package("ops")._SCHEMAS
    assert {name for name, _ in implementations} == {schema.split("(")[0] for schema in schemas}


@pytest.mark.gpu
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs a device that is not the current one")
def test_a_device_that_is_not_current(vgo, device):
    layers = import_package("layers")
    other = torch.device("cuda", 1)
    with torch.cuda.device(0):
        for ours, theirs in zip(layers.rope_sincos(5, 7, 64, device=other), layers.rope_sincos(5, 7, 64)):
            assert ours.device == other
            torch.testing.assert_close(ours.cpu(), theirs, rtol=0, atol=1e-5)
        q, k, v = (torch.randn(1, 2, 70, 64, device=other) for _ in range(3))
        out = vgo.mass_bias_attention(q, k, v, torch.zeros(70, device=other))
        ref = torch.nn.functional.scaled_dot_product_attention(q.double().cpu(), k.double().cpu(), v.double().cpu())
        assert out.device == other
        torch.testing.assert_close(out.cpu().double(), ref, rtol=0, atol=1e-5)
        assert torch.cuda.current_device() == 0
