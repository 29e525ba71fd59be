"""The forward product for few rows per expert: what a row's sum depends on."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native, functions

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


# an expert's rows on both sides of a block's 16, a group's 32 and the next; one, two and (16 bits) four blocks of columns to a workgroup
COUNTS = [1, 0, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130] + [0] * 120


@pytest.mark.parametrize("d,h", [(24, 40), (136, 200), (264, 8200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_inference_and_training_have_the_same_result(d, h, dtype, device):
    """Weights past the caches where nothing is differentiated, through them where a backward will read them: what is read is the same, bit for bit."""
    e, n = len(COUNTS), sum(COUNTS)
    assert n <= 4 * e and 2 * e * d * h < 1 << 30   # (the rule's line; either side of what the caches hold)
    g = torch.Generator().manual_seed(d)
    idx = torch.repeat_interleave(torch.arange(e), torch.tensor(COUNTS))[torch.randperm(n, generator=g)].unsqueeze(1).to(device)
    new = lambda *s: torch.randn(*s, generator=g).to(dtype).to(device)
    x, score, w1, b1, w2, b2 = new(n, d), new(n, 1), new(e, h, d) / d ** 0.5, new(e, h), new(e, d, h) / h ** 0.5, new(e, d)
    counts, pos, slot_to_row = fmoe_native.route(idx, e)
    routing = pos, slot_to_row.view(-1), fmoe_native.segment_table(counts, n)
    args = x, None, None, score, w1, b1, w2, b2, routing, 1, _lib.ACT_RELU, _lib.GATE_ROUTED
    with torch.no_grad():
        once = functions.layer_call(*args)
    w1.requires_grad_(True)
    kept = functions.layer_call(*args)
    assert kept.requires_grad and not once.requires_grad and torch.equal(kept.detach(), once)
    rows = torch.cat([torch.relu(x[t] @ w1[i].t() + b1[i]) @ w2[i].t() + b2[i] for t, i in zip(range(3), idx[:3, 0].tolist())]).view(3, d)
    assert (once[:3] - rows * score[:3]).float().norm() <= 0.02 * (rows * score[:3]).float().norm()
