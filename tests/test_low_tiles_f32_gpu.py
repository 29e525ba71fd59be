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
