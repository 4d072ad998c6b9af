"""The matcher where the source count lives on the device, and on both sides of the size at
which the staged kernel gives way to the ring kernel: bit for bit the results of the same
rows matched on their own, and of torch on the bf16-rounded scores."""
from __future__ import annotations

import ctypes

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


@pytest.mark.parametrize("n_src,n_dict", [(2304, 2304), (2305, 2303), (2303, 2305), (2304, 2177), (2304, 2176),
                                          (2100, 2048 + 64), (5376, 1500)])
def test_half_dictionary_tiles_match_whole_ones(vgo, device, n_src, n_dict):
    """Sizes that take 128-row dictionary tiles, against the device-count launch (256-row tiles)."""
    kern = import_package("_kernels")
    src, dic = _rows(8, n_src, 64, device), _rows(9, n_dict + 40, 64, device)
    dic[1::3] = dic[0]  # ties
    src[5] = float("nan")
    dic[n_dict // 2] = float("nan")
    dic[7, 0] = float("inf")
    rows = torch.randperm(n_src, generator=torch.Generator().manual_seed(10)).to(device)
    rows[11] = -1
    rows[12] = n_src
    index_map = torch.randperm(n_dict + 40, generator=torch.Generator().manual_seed(11)).to(device)
    for clean in (False, True):
        if clean:
            src, dic = src.nan_to_num(0.0), dic.nan_to_num(0.0, 1.0, -1.0)
        options = dict(dict_ranges=(n_dict - 300, n_dict - 260, n_dict), index_map=index_map, src_rows=rows)
        print(f"[match] half tiles {n_src} x {n_dict} clean={clean}", flush=True)
        values, index = kern.similarity_topk(src, dic, 4, **options)
        ref_v, ref_i = torch.empty_like(values), torch.empty_like(index)
        kern.similarity_topk(src, dic, 4, n_src=n_src, out=(ref_v, ref_i), **options,
                             n_src_device=torch.tensor([n_src], dtype=torch.int32, device=device))
        assert torch.equal(index, ref_i) and torch.equal(values.nan_to_num(9.0), ref_v.nan_to_num(9.0))


def test_device_counts_with_the_least_workspace(vgo, device):
    package, kern = import_package("_lib"), import_package("_kernels")
    lib = package.load()
    bound, n_dict, dim, topk, count = 5600, 2800, 64, 4, 1500
    src, dic = _rows(12, bound, dim, device), _rows(13, n_dict, dim, device)
    parts, size = ctypes.c_int(), ctypes.c_size_t()
    package.check(lib.vgo_similarity_topk_workspace(bound, n_dict, topk, ctypes.byref(parts), ctypes.byref(size)))
    least = bound * parts.value * topk * 8
    assert least < size.value
    want_v, want_i = kern.similarity_topk(src[:count], dic, topk)
    for nbytes in (least, size.value):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
        values, index = torch.empty(bound, topk, device=device), torch.empty(bound, topk, device=device, dtype=torch.int64)
        n = torch.tensor([count], dtype=torch.int32, device=device)
        package.check(lib.vgo_similarity_topk(
            src.data_ptr(), dim, bound, None, n.data_ptr(), bound, dic.data_ptr(), dim, n_dict, n_dict, 0, n_dict, dim,
            topk, ws.data_ptr(), nbytes, values.data_ptr(), index.data_ptr(), None, None, None, 0,
            torch.cuda.current_stream(device).cuda_stream))
        assert torch.equal(values[:count], want_v) and torch.equal(index[:count], want_i)
