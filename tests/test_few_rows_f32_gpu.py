"""The forward product for few rows per expert in float32 (weights straight from memory to the matrix pipe)."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu

# blocks of 16 rows, groups of 32, a tile of 128 and the next; experts without rows keep the average below the rule's line
EDGES = [1, 0, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 130] + [0] * 9
# past 1024 experts, which are not in order of their rows: row tiles of 128
TILES = [1, 0, 17, 128, 129, 300] + [0] * 1100 + [33]


# (one block of 16 columns to a workgroup, and two where 22 experts make a workgroup of them for each of 256 compute units)
@pytest.mark.parametrize("k,n", [(4, 4), (16, 16), (20, 36), (68, 20), (256, 64), (1028, 132), (68, 388), (260, 356)])
@pytest.mark.parametrize("act", [_lib.ACT_NONE, _lib.ACT_RELU, _lib.ACT_GELU])
def test_few_rows_in_float32(k, n, act, device):
    against_float64(EDGES, k, n, act, device)


@pytest.mark.parametrize("k,n", [(20, 36), (260, 68)])
def test_few_rows_of_more_experts_than_the_table_sorts(k, n, device):
    against_float64(TILES, k, n, _lib.ACT_RELU, device)


def against_float64(sizes, k, n, act, device):
    """Against float64, element by element: 2 k + 8 roundings of float32 of the terms' absolute sum bound any order of the
    products, the waves' sums and the bias; GELU's own formula is within 1.5e-7 of its argument's size."""
    counts = torch.tensor(sizes)
    e, rows = len(sizes), sum(sizes)
    slots = rows + 5
    assert slots <= 24 * e   # (the rule's line)
    g = torch.Generator().manual_seed(k + n)
    x = torch.randn(slots, k, generator=g).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(device)
    b = torch.randn(e, n, generator=g).to(device)
    table = fmoe_native.segment_table(counts.to(device), slots)
    index = torch.randint(0, 3 * slots, (slots,), generator=g)
    index[torch.rand(slots, generator=g) < 0.1] = -1
    index = index.to(device)
    picked = torch.where(index[:, None] >= 0, x[(index // 3).clamp(min=0)], torch.zeros_like(x))
    for src, kw in ((x, {}), (picked, dict(row_index=index, index_div=3))):
        y, pre = fmoe_native.linear_forward_dev(x, w, b, table, slots, act, act != _lib.ACT_NONE, **kw)
        lo = 0
        for i, c in enumerate(sizes):
            a, we = src[lo:lo + c].double(), w[i].double()
            ref = a @ we.t() + b[i].double()
            bound = (2 * k + 8) * 2.0 ** -24 * (a.abs() @ we.abs().t() + b[i].double().abs())
            got = (pre if pre is not None else y)[lo:lo + c].double()
            assert ((got - ref).abs() <= bound).all()
            if act == _lib.ACT_RELU:
                assert torch.equal(y[lo:lo + c], pre[lo:lo + c].clamp(min=0))
            if act == _lib.ACT_GELU:
                want = torch.nn.functional.gelu(pre[lo:lo + c].double())
                assert ((y[lo:lo + c].double() - want).abs() <= 4e-7 * (1 + pre[lo:lo + c].double().abs())).all()
            lo += c


@pytest.mark.parametrize("act", [_lib.ACT_NONE, _lib.ACT_GELU])
def test_the_rows_past_the_counts_are_left_alone(act, device, monkeypatch):
    """Outputs that begin as a value no product makes still hold it past the counts, bit for bit."""
    counts = torch.tensor([3, 0, 2], device=device)
    table = fmoe_native.segment_table(counts, 64)
    x, w = torch.randn(64, 32, device=device), torch.randn(3, 48, 32, device=device)
    marker = -1.25e33
    real = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: real(*a, **k).fill_(marker) if k.get("dtype") == torch.float32 else real(*a, **k))
    y, pre = fmoe_native.linear_forward_dev(x, w, None, table, 64, act, act != _lib.ACT_NONE)
    ref = torch.cat([x[:3].double() @ w[0].double().t(), x[3:5].double() @ w[2].double().t()])
    full = y if pre is None else pre
    assert (full[:5].double() - ref).abs().max() <= 1e-5 * ref.abs().max()
    for t in (y, pre):
        if t is not None:
            assert t.shape[0] == 64 and (t[:5] != marker).all() and (t[5:] == torch.tensor(marker, device=device)).all()


# (the second: past 1024 experts, and past 4 GiB)
@pytest.mark.parametrize("e,rows", [(1024, 12288), (2048, 24576)])
def test_rows_of_one_expert_past_two_gib(e, rows, device):
    """All rows are one expert's, more than 32-bit offsets reach.  Small whole numbers: sums below 2^24, exact in any order.  The last rows are
    infinite, so that a row which reads them in place of what lies past its contraction is not a number."""
    k, n, one = 43720, 4, e - 3
    assert (1 << 31) * (rows // 12288) < rows * k * 4 and rows <= 12 * e and 6 * k < 1 << 24
    g = torch.Generator(device=device).manual_seed(e)
    x = torch.empty(rows, k, device=device)
    for part in x.split(2048):
        part.copy_(torch.randint(-1, 3, part.shape, device=device, generator=g, dtype=torch.int8))
    x[-8:] = float("inf")
    w = torch.zeros(e, n, k, device=device)
    w[one] = torch.randint(-3, 4, (n, k), device=device, generator=g).float()
    counts = torch.zeros(e, dtype=torch.int64)
    counts[one] = rows
    table = fmoe_native.segment_table(counts.to(device), rows)
    y = fmoe_native.linear_forward_dev(x, w, None, table, rows)[0]
    for got, part in zip(y[:-8].split(2048), x[:-8].split(2048)):
        assert torch.equal(got, (part.double() @ w[one].double().t()).float())
