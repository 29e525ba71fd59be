"""Products over a device table whose weights are read past the caches, where the average expert has one row tile."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu


def operands(counts, k, n, dtype, device):
    rows = sum(counts)
    g = torch.Generator(device=device).manual_seed(k + rows)
    new = lambda *s: torch.randn(*s, generator=g, device=device).to(dtype)
    return new(rows, k), new(len(counts), n, k) / k ** 0.5, new(len(counts), n), new(rows, n)


# (loads past the caches begin at weights of 128 MiB)
@pytest.mark.parametrize("tile", ["64x128", "128x128", "128x128+", "128x256", "256x256"])
@pytest.mark.parametrize("counts", [[3, 0, 40, 17], [49, 50, 1, 0], [219, 219, 219, 220]])
def test_results_with_large_weights(tile, counts, device, monkeypatch):
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    k, n = 4104, 4168
    x, w, b, gy = operands(counts, k, n, torch.bfloat16, device)
    assert w.numel() * 2 > 128 << 20
    host = torch.tensor(counts)
    table = fmoe_native.segment_table(host.to(device), sum(counts))
    y, pre = fmoe_native.linear_forward_dev(x, w, b, table, sum(counts), _lib.ACT_GELU, True)
    ref, ref_pre = fmoe_native.linear_act_forward(x, host, w, b, _lib.ACT_GELU)
    gx, ref_gx = fmoe_native.linear_dgrad_dev(gy, w, table, sum(counts)), fmoe_native.linear_backward(gy, x, host, w, b)[0]
    # (the host's launches may split a tail's contraction: its terms in another order, 4168 roundings of 2^-24 at most, and one of 2^-8)
    for got, want in ((pre, ref_pre), (y, ref), (gx, ref_gx)):
        assert (got.float() - want.float()).norm() <= 2.0 ** -8 * want.float().norm()


# few experts with small weights, which are read through the caches however many rows there are
@pytest.mark.parametrize("tile", ["64x128", "128x128", "128x128+", "128x256", "256x256"])
@pytest.mark.parametrize("counts", [[3, 0, 40, 17], [300, 1, 0, 2], [108, 110, 109, 110], [219, 219, 219, 220], [256, 255, 257, 300]])
@pytest.mark.parametrize("k,n", [(64, 256), (200, 136)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_results_are_those_of_the_host_counts(tile, counts, k, n, dtype, device, monkeypatch):
    """Launches over a device table and from host counts, both through the caches: bit for bit the same."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    e, rows = len(counts), sum(counts)
    g = torch.Generator().manual_seed(k + rows)
    x = torch.randn(rows, k, generator=g).to(dtype).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(dtype).to(device)
    b = torch.randn(e, n, generator=g).to(dtype).to(device)
    gy = torch.randn(rows, n, generator=g).to(dtype).to(device)
    host = torch.tensor(counts)
    table = fmoe_native.segment_table(host.to(device), rows)
    y, pre = fmoe_native.linear_forward_dev(x, w, b, table, rows, _lib.ACT_GELU, True)
    ref, ref_pre = fmoe_native.linear_act_forward(x, host, w, b, _lib.ACT_GELU)
    assert torch.equal(y, ref) and torch.equal(pre, ref_pre)
    gx = fmoe_native.linear_dgrad_dev(gy, w, table, rows)
    assert torch.equal(gx, fmoe_native.linear_backward(gy, x, host, w, b)[0])


# weights of 131 MiB; at most 6/7 of a tile's height per expert on average, so that all five tiles read past the caches, and more, so that the lower do not
@pytest.mark.parametrize("tile", ["64x128", "128x128", "128x128+", "128x256", "256x256"])
@pytest.mark.parametrize("counts", [[3, 0, 40, 17], [130, 1, 0, 2], [70, 66, 1, 90]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_loads_past_the_caches_read_the_same(tile, counts, dtype, device, monkeypatch):
    """Where a load leaves traces makes no difference to what it reads: bit for bit the launch from host counts, which reads through the caches
    (contractions of 17 slabs, which no launch splits), with rows in order and through an index, plain and with the activation's derivative."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    counts = counts * 16
    e, rows, k, n = len(counts), sum(counts), 1032, 1040
    assert e * k * n * 2 > 128 << 20
    x, w, b, gy = operands(counts, k, n, dtype, device)
    pre_in = torch.randn(rows, k, device=device).to(dtype)
    host = torch.tensor(counts)
    table = fmoe_native.segment_table(host.to(device), rows)
    y, pre = fmoe_native.linear_forward_dev(x, w, b, table, rows, _lib.ACT_GELU, True)
    ref, ref_pre = fmoe_native.linear_act_forward(x, host, w, b, _lib.ACT_GELU)
    assert torch.equal(y, ref) and torch.equal(pre, ref_pre)
    index = torch.randperm(3 * rows, device=device)[:rows]
    y = fmoe_native.linear_forward_dev(x, w, b, table, rows, _lib.ACT_GELU, True, row_index=index, index_div=3)[0]
    assert torch.equal(y, fmoe_native.linear_act_forward(x[index // 3].contiguous(), host, w, b, _lib.ACT_GELU)[0])
    assert torch.equal(fmoe_native.linear_dgrad_dev(gy, w, table, rows), fmoe_native.linear_backward(gy, x, host, w, b)[0])
    for act in (_lib.ACT_RELU, _lib.ACT_GELU):
        assert torch.equal(fmoe_native.linear_dgrad_dev(gy, w, table, rows, pre_in, act), fmoe_native.linear_dact_backward(gy, host, w, pre_in, act))
