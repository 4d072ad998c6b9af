"""Inputs of the restore map that its kernel would read out of range, or in host memory, are refused before it runs."""
from __future__ import annotations

import pytest
import torch

from tests.conftest import import_package


def _restore_map(*args, **kwargs):
    import_package("_lib").load()
    return import_package("_kernels").restore_map(*args, **kwargs)


def test_host_tensors_are_refused():
    with pytest.raises(RuntimeError, match="vgo kernels run on the GPU only"):
        _restore_map(4, device="cpu", inverse=torch.zeros(4, dtype=torch.int64))


@pytest.mark.gpu
def test_short_and_host_operands(vgo, device):
    ids = torch.arange(4, device=device)
    with pytest.raises(ValueError, match="4 inverse entries for 5 tokens"):
        _restore_map(5, device=device, inverse=ids)
    with pytest.raises(ValueError, match="four parents"):
        _restore_map(8, device=device, keep=ids, source=ids + 4, parent=ids.repeat(3), weight=torch.ones(16, device=device))
    with pytest.raises(RuntimeError, match="GPU only"):
        _restore_map(8, device=device, keep=ids, source=ids + 4, parent=ids.repeat(4), weight=torch.ones(16))
    index, weight = _restore_map(8, device=device, keep=ids, source=ids + 4, parent=ids.repeat(4),
                                 weight=torch.ones(16, device=device))
    assert torch.equal(index[:4, 0].long(), ids) and torch.equal(weight[4:], torch.ones(4, 4, device=device))
    assert torch.equal(_restore_map(3, device=device, inverse=ids)[0][:, 0].long(), ids[:3])  # a longer one's first
    with pytest.raises(RuntimeError, match="GPU only"):  # the mass of host weights
        vgo.deterministic_weighted_normalizer(ids.view(1, 1, 4), torch.ones(1, 1, 4), 4)
