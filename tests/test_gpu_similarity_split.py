"""The matcher where the source count lives on the device, and on both sides of the size at
which the staged kernel gives way to the ring kernel: bit for bit the results of the same
rows matched on their own, and of torch on the bf16-rounded scores."""
from __future__ import annotations

import pytest
import torch

from tests.conftest import import_package

pytestmark = pytest.mark.gpu


def _rows(seed, n, dim, device):
    g = torch.Generator(device=device).manual_seed(seed)
    return torch.nn.functional.normalize(torch.randn(n, dim, generator=g, device=device), dim=1).bfloat16()


@pytest.mark.parametrize("topk", [1, 4])
@pytest.mark.parametrize("bound,n_dict,dim", [(700, 900, 64), (2100, 2300, 64), (33000, 520, 32), (600, 300, 72)])
def test_device_counts_match_host_counts(vgo, device, topk, bound, n_dict, dim):
    kern = import_package("_kernels")
    src, dic = _rows(1, bound, dim, device), _rows(2, n_dict, dim, device)
    rows = torch.randperm(bound, generator=torch.Generator().manual_seed(3)).to(device)
    for count in sorted({0, 1, 127, 129, 256, 257, bound // 3, bound - 1, bound}):
        print(f"[match] topk={topk} bound={bound} count={count}", flush=True)
        values = torch.full((bound, topk), 7.0, device=device)
        index = torch.full((bound, topk), -7, device=device)
        kern.similarity_topk(src, dic, topk, src_rows=rows, n_src=bound, out=(values, index),
                             n_src_device=torch.tensor([count], dtype=torch.int32, device=device))
        if count:
            ref_v, ref_i = kern.similarity_topk(src[rows[:count]], dic, topk)
            assert torch.equal(values[:count], ref_v) and torch.equal(index[:count], ref_i)
        assert bool((values[count:] == 7.0).all()) and bool((index[count:] == -7).all())


@pytest.mark.parametrize("n_src,n_dict", [(2048, 2048), (2049, 2048), (256, 16384), (256, 16385)])
def test_staged_and_ring_kernels_agree_at_their_border(vgo, device, n_src, n_dict):
    kern = import_package("_kernels")
    src, dic = _rows(5, n_src, 96, device), _rows(6, n_dict, 96, device)
    v1, i1 = kern.similarity_topk(src, dic, 1)
    v4, i4 = kern.similarity_topk(src, dic, 4)
    # The same rows as part of a larger problem run on the ring kernel.
    big_v, big_i = kern.similarity_topk(torch.cat((src, _rows(7, 4096, 96, device))), dic, 4)
    assert torch.equal(v4, big_v[:n_src]) and torch.equal(i4, big_i[:n_src])
    assert torch.equal(v1, v4[:, :1]) and torch.equal(i1, i4[:, :1])
