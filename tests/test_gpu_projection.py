"""Parity of the gfx950 top-4 projection kernel against the CPU oracle.

The kernel and the oracle perform the same IEEE operations in the same order
(weight rounded to the value type, each product rounded, fp32 sum in corner
order), so the comparison is bit-exact.
"""
from __future__ import annotations

import pytest
import torch

from oracle import projection as oracle

pytestmark = pytest.mark.gpu


def _case(seed, n, m, d, dtype):
    g = torch.Generator().manual_seed(seed)
    table = torch.randn(m, d, generator=g).to(dtype)
    keys = torch.rand(n, m, generator=g) if m <= 4096 else None
    if keys is not None:
        index = keys.argsort(dim=1)[:, :4].int()
    else:
        index = torch.randint(0, m, (n, 4), generator=g, dtype=torch.int32)
    e = -torch.rand(n, 4, generator=g, dtype=torch.float64).log()
    weight = (e / e.sum(1, keepdim=True)).float()
    return table, index, weight


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("n,m,d", [(1, 4, 8), (97, 31, 64), (1044, 522, 1024), (333, 50, 1000),
                                   (4099, 700, 2048), (257, 16, 23)])
def test_bit_exact_vs_oracle(vgo, device, dtype, n, m, d):
    print(f"[project] dtype={dtype} n={n} m={m} d={d}", flush=True)
    table, index, weight = _case(n + m + d, n, m, d, dtype)
    out = vgo.top4_project(table.to(device), index.to(device), weight.to(device))
    torch.cuda.synchronize()
    ref = oracle.top4_project(table, index, weight)
    assert torch.equal(out.cpu(), ref)


def test_one_hot_restore_is_exact_copy(vgo, device):
    table, index, _ = _case(3, 500, 200, 1024, torch.bfloat16)
    weight = torch.zeros(index.shape)
    weight[:, 0] = 1.0
    out = vgo.top4_project(table.to(device), index.to(device), weight.to(device))
    assert torch.equal(out.cpu(), table[index[:, 0].long()])


def test_bad_index_poisons_row_without_reading(vgo, device):
    table, index, weight = _case(4, 64, 32, 256, torch.float32)
    index[3, 2] = 1 << 30
    index[9, 1] = -5
    weight[9, 1] = 0.0
    out = vgo.top4_project(table.to(device), index.to(device), weight.to(device)).cpu()
    assert torch.isnan(out[3]).all()
    assert torch.isfinite(out[9]).all()
    ref = oracle.top4_project(table, index, weight)
    assert torch.equal(torch.nan_to_num(out), torch.nan_to_num(ref))


def test_strided_table_and_output(vgo, device):
    table, index, weight = _case(6, 300, 90, 512, torch.bfloat16)
    wide = torch.zeros(90, 1024, dtype=torch.bfloat16)
    wide[:, 256:768] = table
    out = torch.full((300, 1024), 7.0, dtype=torch.bfloat16, device=device)
    view = out[:, 128:640]
    vgo.top4_project(wide.to(device)[:, 256:768], index.to(device), weight.to(device), out=view)
    ref = oracle.top4_project(table, index, weight)
    assert torch.equal(view.cpu(), ref)
    assert (out[:, :128] == 7).all() and (out[:, 640:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,m,d", [(4099, 700, 1024), (1044, 522, 1000), (257, 16, 23)])
def test_ordered_projection_equals_plain(dtype, device, n, m, d):
    """Rows computed in the locality order (grouped by first parent) or any other
    order give the plain projection bit for bit; order entries outside [0, N)
    compute nothing."""
    print(f"[project] ordered dtype={dtype} n={n} m={m} d={d}", flush=True)
    from tests.conftest import import_package
    proj = import_package("projection")
    table, index, weight = _case(n * 3 + m + d, n, m, d, dtype)
    table, index, weight = table.to(device), index.to(device), weight.to(device)
    plain = proj.top4_project(table, index, weight)
    order = proj.locality_order(index, m)
    assert order.dtype == torch.int32 and torch.equal(order.sort().values.cpu(), torch.arange(n, dtype=torch.int32))
    first = index[:, 0].long()[order.long()].cpu()
    assert bool((first[1:] >= first[:-1]).all()), "locality order must group rows by first parent"
    assert torch.equal(proj.top4_project(table, index, weight, order=order), plain)
    shuffled = torch.randperm(n, generator=torch.Generator().manual_seed(n)).int().to(device)
    assert torch.equal(proj.top4_project(table, index, weight, order=shuffled), plain)
    partial = shuffled.clone()
    partial[: n // 2] = -1
    out = torch.full_like(plain, 7.0)
    proj.top4_project(table, index, weight, out=out, order=partial)
    done = torch.zeros(n, dtype=torch.bool)
    done[partial[n // 2:].long().cpu()] = True
    assert torch.equal(out[done.to(device)], plain[done.to(device)])
    assert bool((out[~done.to(device)] == 7.0).all())


@pytest.mark.parametrize("dtype,n,m,d,strided", [
    (torch.bfloat16, 40007, 3000, 1024, False), (torch.float32, 33001, 1500, 1024, False),
    (torch.float16, 33000, 2500, 1024, True), (torch.bfloat16, 33000, 2500, 1024, True),
    (torch.bfloat16, 32800, 1100, 2048, False)])
def test_large_tables_bit_exact(vgo, device, dtype, n, m, d, strided):
    """Tables larger than an XCD's L2 (4 MB) with tens of thousands of rows, the C2
    regime at a size the oracle checks whole: bit-exact on a ragged row count, strided
    table and output views, a poisoned row (out-of-range id with a non-zero weight), a
    zero-weight out-of-range id that must not poison, and one-hot rows."""
    print(f"[project] large table dtype={dtype} n={n} m={m} d={d} strided={strided}", flush=True)
    table, index, weight = _case(n + m + d, n, m, d, dtype)
    index[5, 1] = m + 17           # poisons row 5
    index[11, 3] = -2              # zero weight: ignored
    weight[11, 3] = 0.0
    weight[13] = torch.tensor([0.0, 1.0, 0.0, 0.0])   # one-hot row
    assert table.numel() * table.element_size() > 4 << 20
    if strided:
        wide = torch.zeros(m, d + 256, dtype=dtype)
        wide[:, 128:128 + d] = table
        table_d = wide.to(device)[:, 128:128 + d]
        out_full = torch.full((n, d + 64), 3.0, dtype=dtype, device=device)
        out = out_full[:, 64:]
    else:
        table_d = table.to(device)
        out_full = out = torch.empty(n, d, dtype=dtype, device=device)
    vgo.top4_project(table_d, index.to(device), weight.to(device), out=out)
    torch.cuda.synchronize()
    got = out.cpu()
    ref = oracle.top4_project(table, index, weight)
    assert torch.isnan(got[5]).all() and torch.isfinite(got[11]).all()
    assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(ref))
    assert torch.equal(got[13], table[index[13, 1].long()])
    if strided:
        assert bool((out_full[:, :64] == 3.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gather_probe_sums_the_projection_rows(vgo, device, dtype):
    """vgo_top4_gather_probe reads what the projection reads and writes each row's sum:
    the sums equal the projection's rows summed (fp32, within summation-order
    rounding), a poisoned row gives NaN in both, and rows of odd width are refused."""
    print(f"[project] gather probe dtype={dtype}", flush=True)
    from tests.conftest import import_package
    proj = import_package("projection")
    table, index, weight = _case(21, 5000, 700, 1024, dtype)
    index[7, 2] = 1 << 20
    td, idd, wd = table.to(device), index.to(device), weight.to(device)
    sums = proj.gather_probe(td, idd, wd)
    rows = proj.top4_project(td, idd, wd).double().sum(1)
    assert torch.isnan(sums[7]) and torch.isnan(rows[7])
    ok = ~torch.isnan(rows)
    assert torch.allclose(sums[ok].double(), rows[ok], rtol=1e-5, atol=1e-3)
    small = table[:, :23].contiguous().to(device)
    with pytest.raises(RuntimeError, match="16-byte"):
        proj.gather_probe(small, idd, wd)


@pytest.mark.parametrize("m", [16384, 16385, 98304, 98305])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_column_slices_at_their_edges(vgo, device, dtype, m):
    """Row counts around a unit of every slice width (4 to 16 rows), and channel counts
    that end inside a slice or give the eight XCDs unequal shares of the slices, on both
    sides of the table sizes at which the slice width and the grid change: bit-exact."""
    for n, d in [(1, 8), (3, 72), (15, 200), (17, 264), (129, 776), (4099, 72)]:
        print(f"[project] slices dtype={dtype} n={n} m={m} d={d}", flush=True)
        table, index, weight = _case(n + m + d, n, m, d, dtype)
        index[0] = torch.tensor([0, m - 1, m - 1, 0], dtype=torch.int32)
        out = vgo.top4_project(table.to(device), index.to(device), weight.to(device))
        assert torch.equal(out.cpu(), oracle.top4_project(table, index, weight))


def _rows_like(pattern, n, m, device, seed):
    """Index and weight of n rows: `kept` and `one_hot` with one corner each (ascending, scattered),
    `part` half and half with four, `near` four corners within 128 table rows, `mixed` four anywhere."""
    g = torch.Generator(device=device).manual_seed(seed)
    ascending = (torch.arange(n, device=device) * m // n)[:, None]
    index = torch.randint(0, m, (n, 4), device=device, generator=g)
    weight = torch.rand(n, 4, device=device, generator=g) + 0.01
    single = torch.zeros(n, dtype=torch.bool, device=device)
    if pattern == "near":
        index = (ascending + torch.randint(-64, 65, (n, 4), device=device, generator=g)).clamp_(0, m - 1)
    if pattern in ("kept", "one_hot", "part"):
        single = torch.rand(n, device=device, generator=g) < 0.5 if pattern == "part" else ~single
        if pattern != "one_hot":
            index[single] = ascending.expand(-1, 4)[single]
        weight[single] = torch.tensor([1.0, 0.0, 0.0, 0.0], device=device)
    weight /= weight.sum(1, keepdim=True)
    index[1], weight[1] = m + 7, 0.25           # poisons its row
    index[n - 1, 3], weight[n - 1, 3] = -3, 0.0  # no weight: ignored
    return index.int(), weight


# On both sides of the output sizes (96, 256, 512 MB and 1.5 GB), the table sizes (12 MB per slice) and
# the row lengths (2, 3 and 4 chunks per lane, the last one ragged) at which whole rows come in.
@pytest.mark.parametrize("dtype,n,m,d", [
    (torch.float32, 24575, 12288, 1024), (torch.float32, 24577, 12288, 1024), (torch.float32, 24577, 49153, 1024),
    (torch.float32, 32901, 60000, 768), (torch.float32, 131075, 49153, 512), (torch.float32, 393217, 49152, 1024),
    (torch.bfloat16, 131073, 3000, 1024), (torch.bfloat16, 43401, 98305, 1160),
    (torch.bfloat16, 262145, 16384, 1024), (torch.bfloat16, 786433, 98304, 1024),
    (torch.float16, 131073, 98305, 1000), (torch.float16, 24577, 9000, 2048),
    (torch.float16, 262145, 98305, 1024), (torch.float16, 786433, 98305, 1024)])
def test_whole_rows_equal_slices(vgo, device, dtype, n, m, d):
    """Rows of every kind that the sample tells apart: the whole call, the rows in an order and the
    same rows in pieces (below 64 MB: by slices) are equal bit for bit, and 256 rows equal the oracle."""
    from tests.conftest import import_package
    proj = import_package("projection")
    table = torch.randn(m, d, device=device, generator=torch.Generator(device=device).manual_seed(n)).to(dtype)
    order = torch.arange(n - 1, -1, -1, dtype=torch.int32, device=device)
    piece = (64 << 20) // (d * table.element_size())
    pick = torch.linspace(0, n - 1, 256).long()
    for pattern in ("kept", "one_hot", "part", "near", "mixed"):
        print(f"[project] {pattern} rows dtype={dtype} n={n} m={m} d={d}", flush=True)
        index, weight = _rows_like(pattern, n, m, device, n + m)
        out = torch.full((n, d), 7.0, dtype=dtype, device=device)
        vgo.top4_project(table, index, weight, out=out)
        assert bool(torch.isnan(out[1]).all()) and bool(torch.isfinite(out[n - 1]).all())
        for r0 in range(0, n, piece):
            part = proj.top4_project(table, index[r0:r0 + piece], weight[r0:r0 + piece])
            assert bool(torch.eq(out[r0:r0 + piece].nan_to_num_(3.0), part.nan_to_num_(3.0)).all()), r0
        assert bool(torch.eq(proj.top4_project(table, index, weight, order=order).nan_to_num_(3.0), out).all())
        used = index[pick.to(device)].clamp(0, m - 1).long()
        ref = oracle.top4_project(table[used.flatten()].cpu(), torch.arange(1024, dtype=torch.int32).view(256, 4),
                                  weight[pick.to(device)].cpu())
        assert torch.equal(out[pick.to(device)].cpu(), ref)
