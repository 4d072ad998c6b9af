"""Corner CSR, plan assembly and failed-row list of the convex planner at the edges of their
chunks and rules, against the plain definitions on the CPU (whole numbers: equal)."""
from __future__ import annotations

import pytest
import torch

from tests.conftest import import_package

pytestmark = pytest.mark.gpu


# 12,288 items and 40,960 buckets are the largest of the one-launch CSR, 4,096 items of its small instance.
@pytest.mark.parametrize("corners", [1, 4])
@pytest.mark.parametrize("items,buckets", [(4, 4), (4096, 1204), (4100, 40960), (12288, 40960), (12288, 40964),
                                           (12292, 8), (12284, 4), (70000, 300)])
@pytest.mark.parametrize("spread", ["random", "skewed", "one"])
def test_corner_csr(vgo, device, items, buckets, corners, spread):
    kern = import_package("_kernels")
    g = torch.Generator().manual_seed(items + buckets + corners)
    dests = buckets // corners
    parent = torch.randint(-1, dests + 1, (items // corners, corners), generator=g)
    if spread == "one":
        parent[:] = dests // 2
    elif spread == "skewed":
        parent[torch.rand(parent.shape, generator=g) < 0.5] = 0
        parent[torch.rand(parent.shape, generator=g) < 0.25] = -(1 << 40)
    print(f"[csr] items={items} buckets={buckets} corners={corners} {spread}", flush=True)
    key = torch.where((parent >= 0) & (parent < dests), parent * corners + torch.arange(corners), buckets).reshape(-1)
    want = key.argsort(stable=True).int()
    want_offsets = torch.cat((torch.zeros(1, dtype=torch.int64),
                              torch.bincount(key, minlength=buckets + 1)[:buckets].cumsum(0))).int()
    order, offsets = kern.corner_csr(parent.to(device), dests)
    assert torch.equal(order.cpu(), want) and torch.equal(offsets.cpu(), want_offsets)
    order, offsets = kern.csr_build(key.to(device), buckets)
    assert torch.equal(order.cpu(), want) and torch.equal(offsets.cpu(), want_offsets)


# 1,024 elements per chunk, 65,536 per group of chunks.
@pytest.mark.parametrize("n,total", [(0, 0), (0, 5), (1, 1), (1023, 1024), (1025, 2049), (6500, 8700), (65536, 65537),
                                     (70000, 131073)])
def test_assemble_and_failed_rows(vgo, device, n, total):
    package = import_package("_lib")
    lib = package.load()
    g = torch.Generator().manual_seed(n + total)
    candidate = torch.randperm(max(total, 1), generator=g)[:n].sort().values
    fit, top1 = torch.rand(n, generator=g), torch.rand(n, generator=g)
    fit[::7] = float("nan")
    fit[1::7] = 0.5
    alpha = torch.rand((n, 4), generator=g)
    support = torch.randint(-1, total + 1, (n, 4), generator=g)
    threshold, easy = 0.5, 0.625
    selected = fit >= threshold
    hard = ~(top1 >= easy)
    failed = (hard & (fit < threshold)).nonzero().flatten().int()
    source = candidate[selected]
    o2c = torch.ones(total, dtype=torch.int64)
    o2c[source] = 0
    keep = o2c.nonzero().flatten()
    o2c = torch.where(o2c == 1, o2c.cumsum(0) - 1, -1)
    sup = support[selected]
    parent = torch.where((sup >= 0) & (sup < total), o2c[sup.clamp(0, max(total - 1, 0))] if total else sup, -1)

    dev = {k: v.to(device) for k, v in dict(fit=fit, alpha=alpha, support=support, candidate=candidate,
                                            top1=top1).items()}
    full = lambda shape, dtype: torch.full(shape, 77, device=device, dtype=dtype)  # noqa: E731
    got_list, got_count = full((max(n, 1),), torch.int32), full((1,), torch.int32)
    got = dict(keep=full((total + 1,), torch.int64), o2c=full((total + 1,), torch.int64),
               source=full((n + 1,), torch.int64), parent=full((n + 1, 4), torch.int64),
               weight=full((n + 1, 4), torch.float32), stats=full((4,), torch.float32))
    stream = torch.cuda.current_stream(device).cuda_stream
    print(f"[assemble] n={n} total={total}", flush=True)
    if n:
        package.check(lib.vgo_failed_rows(dev["fit"].data_ptr(), dev["top1"].data_ptr(), easy, n, threshold,
                                          got_list.data_ptr(), got_count.data_ptr(), stream))
        assert int(got_count) == len(failed) and torch.equal(got_list[:len(failed)].cpu(), failed)
    package.check(lib.vgo_sparse_convex_assemble(
        dev["fit"].data_ptr(), dev["alpha"].data_ptr(), dev["support"].data_ptr(), dev["candidate"].data_ptr(),
        dev["top1"].data_ptr(), easy, got_count.data_ptr(), n, total, threshold,
        *(got[k].data_ptr() for k in ("keep", "o2c", "source", "parent", "weight", "stats")), stream))
    got = {k: v.cpu() for k, v in got.items()}
    m = len(source)
    for name, want in (("keep", keep), ("o2c", o2c), ("source", source), ("parent", parent),
                       ("weight", alpha[selected])):
        assert torch.equal(got[name][:len(want)], want), name
        assert bool((got[name][max(len(want), m):][-1:] == 77).all()), f"{name}: written past its end"
    assert got["stats"][:3].tolist() == [m, int(hard.sum()), int(got_count)]
    # fp32 sums of m terms in any order: m * 2^-24 * sum bounds the error.
    exact = float(fit[selected].double().sum())
    assert abs(float(got["stats"][3]) - exact) <= m * 2.0 ** -24 * exact
