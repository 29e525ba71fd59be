"""float32 row tiles of at most half their rows: what a full tile gives for the same rows, bit by bit."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", ["128x128", "128x128+"])
@pytest.mark.parametrize("rest", [1, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("k,n", [(4, 4), (100, 260), (512, 392)])
def test_rows_of_a_low_tile(rest, k, n, tile, device, monkeypatch):
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    g = torch.Generator().manual_seed(rest + k)
    x, w = torch.randn(rest, k, generator=g), torch.randn(1, n, k, generator=g)
    gy, pre = torch.randn(rest, n, generator=g), torch.randn(rest, k, generator=g)
    x[0, :4] = 2.0 ** -100   # (k 4: a row with which the tile goes to the fp32 instruction)
    bias = torch.randn(1, n, generator=g).to(device)
    results = []
    for more in (0, 128 - rest):   # the same rows alone and with others after them in their tile
        def fill(t):
            return torch.cat([t, torch.randn(more, t.shape[1], generator=g)]).to(device)
        rows = rest + more
        table = fmoe_native.segment_table(torch.tensor([rows]).to(device), rows)
        xs, gys = fill(x), fill(gy)
        y, aux = fmoe_native.linear_forward_dev(xs, w.to(device), bias, table, rows, _lib.ACT_GELU, True)
        plain = fmoe_native.linear_forward_dev(xs, w.to(device), None, table, rows)[0]
        gx = fmoe_native.linear_dgrad_dev(gys, w.to(device), table, rows, fill(pre), _lib.ACT_RELU)
        results.append([t[:rest] for t in (y, aux, plain, gx)])
    for low, full in zip(*results):
        assert torch.equal(low, full)


# lanes hold experts i, 64 + i, ..: up to four to a lane, and past 256 the table's own order
@pytest.mark.parametrize("e", [65, 130, 256, 257])
@pytest.mark.parametrize("tile", ["128x128", "128x128+"])
def test_low_tiles_of_many_experts(e, tile, device, monkeypatch):
    """Over a device table, where low tiles come last, what the launch from host counts gives, bit by bit (a contraction that no launch splits); and
    against float64: 2 k + 8 roundings of the terms' absolute sum."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    k, n = 68, 132
    g = torch.Generator().manual_seed(e)
    counts = torch.randint(0, 300, (e,), generator=g)
    counts[::7] = 0
    counts[3::11] = 128
    counts[63], counts[64], counts[-1] = 1, 65, 193
    rows = int(counts.sum())
    x, gy, pre = torch.randn(rows, k, generator=g).to(device), torch.randn(rows, n, generator=g).to(device), torch.randn(rows, k, generator=g).to(device)
    w, b = torch.randn(e, n, k, generator=g).to(device), torch.randn(e, n, generator=g).to(device)
    table = fmoe_native.segment_table(counts.to(device), rows)
    y = fmoe_native.linear_forward_dev(x, w, b, table, rows)[0]
    assert torch.equal(y, fmoe_native.linear_forward(x, counts, w, b))
    gx = fmoe_native.linear_dgrad_dev(gy, w, table, rows, pre, _lib.ACT_RELU)
    assert torch.equal(gx, fmoe_native.linear_dact_backward(gy, counts, w, pre, _lib.ACT_RELU))
    for i, (part, got) in enumerate(zip(x.split(counts.tolist()), y.split(counts.tolist()))):
        ref, mag = part.double() @ w[i].double().t() + b[i].double(), part.double().abs() @ w[i].double().abs().t() + b[i].double().abs()
        assert ((got.double() - ref).abs() <= (2 * k + 8) * 2.0 ** -24 * mag).all()
