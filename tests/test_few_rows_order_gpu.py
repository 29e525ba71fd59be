"""The forward product for few rows per expert: what a row's sum depends on."""
import pytest
import torch

from fastermoe_amd import fmoe_native

pytestmark = pytest.mark.gpu


# (16, 32 and, in 16 bits, 64 columns to a workgroup: 24 experts on 256 compute units)
@pytest.mark.parametrize("k,n", [(2056, 40), (1032, 520), (520, 8200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_a_row_has_the_same_sum_whatever_the_other_experts_have(k, n, dtype, device):
    """The same rows of one expert, few, some and many of them, among others whose rows place the expert first, last or between in the table's order:
    bit for bit the same.  Rows of one expert that are alike have the same result wherever they stand, in groups of 32 too."""
    e, cap, mine = 24, 96, 7   # (four rows per expert on average: this kernel's)
    g = torch.Generator().manual_seed(k)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(dtype).to(device)
    b = torch.randn(e, n, generator=g).to(dtype).to(device)
    for rows in (3, 20, 40):
        x = torch.randn(rows, k, generator=g).to(dtype)
        x[rows - 1] = x[0]   # (of 40 in the second group)
        results = []
        for others in ([0] * e, [1] * e, [2] * 12 + [1] * 12, [0] * 5 + [45] + [0] * 18, [0] * 20 + [11] * 4):
            counts = torch.tensor(others)
            counts[mine] = rows
            assert counts.sum() <= cap
            lo = int(counts[:mine].sum())
            full = torch.randn(cap, k, generator=g).to(dtype)
            full[lo:lo + rows] = x
            table = fmoe_native.segment_table(counts.to(device), cap)
            results.append(fmoe_native.linear_forward_dev(full.to(device), w, b, table, cap)[0][lo:lo + rows])
        for other in results[1:]:
            assert torch.equal(other, results[0])
        assert torch.equal(results[0][0], results[0][rows - 1])
