"""The forward product for few rows per expert in 16-bit types (weights straight from memory to the matrix pipe)."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu

# eight and sixteen rows to a load and a block, passes of 32, a tile of 128 and the next; experts without rows keep the average below
# the rule's line
EDGES = [1, 0, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130] + [0] * 120
FEW = [1, 0, 2]
MANY = [1, 0, 17, 40] + [0] * 1100 + [33]   # past 1024 experts, which are not in order of their rows
TILES = [128, 129, 0, 300] + [0] * 1100 + [1, 256]   # there: experts of one row tile and of several


# one, two and four blocks of 16 columns to a workgroup; contractions that end inside a line of 128 bytes, a unit, a turn of the waves
@pytest.mark.parametrize("k,n,counts", [(8, 16, FEW), (264, 40, FEW), (72, 24, EDGES), (136, 200, EDGES), (1032, 264, EDGES), (520, 8200, FEW),
                                        (200, 8136, EDGES), (72, 24, MANY), (72, 72, TILES)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_rows_in_16_bits(k, n, counts, dtype, device):
    """Against float64, element by element: 2 k + 8 roundings of float32 of the terms' absolute sum bound any order of the products,
    the waves' sums and the bias, and the result is rounded once to the type (half a step, up to 2^-8 or 2^-11 of its size)."""
    e, rows = len(counts), sum(counts)
    slots = rows + 3
    assert slots <= 4 * e   # (the rule's line)
    g = torch.Generator().manual_seed(k + n)
    x = torch.randn(slots, k, generator=g).to(dtype).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(dtype).to(device)
    b = torch.randn(e, n, generator=g).to(dtype).to(device)
    table = fmoe_native.segment_table(torch.tensor(counts).to(device), slots)
    index = torch.randint(0, 3 * slots, (slots,), generator=g)
    index[torch.rand(slots, generator=g) < 0.1] = -1
    index = index.to(device)
    picked = torch.where(index[:, None] >= 0, x[(index // 3).clamp(min=0)], torch.zeros_like(x))
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for src, kw in ((x, {}), (picked, dict(row_index=index, index_div=3))):
        y, pre = fmoe_native.linear_forward_dev(x, w, b, table, slots, _lib.ACT_RELU, True, **kw)
        lo = 0
        for i, c in enumerate(counts):
            a, we = src[lo:lo + c].double(), w[i].double()
            ref = a @ we.t() + b[i].double()
            bound = (2 * k + 8) * 2.0 ** -24 * (a.abs() @ we.abs().t() + b[i].double().abs())
            got = pre[lo:lo + c].double()
            assert ((got - ref).abs() <= bound * (1 + step) + step * ref.abs() + 2.0 ** -24).all()   # (the last: denormal halves)
            assert torch.equal(y[lo:lo + c], pre[lo:lo + c].clamp(min=0))
            lo += c
