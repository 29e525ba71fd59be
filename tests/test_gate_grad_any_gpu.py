"""The gate's gradients in 16-bit types whose rows are no whole 16-byte chunks."""
import pytest
import torch

from fastermoe_amd import fmoe_native

pytestmark = pytest.mark.gpu
STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # half a rounding step of the type, of a value just above a power of two


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,e,k", [(1, 1, 1, 1), (5, 7, 3, 2), (64, 9, 16, 1), (130, 127, 17, 4), (777, 500, 12, 2), (65, 1031, 70, 8), (200, 4093, 256, 1)])
def test_against_float64(n, d, e, k, dtype, device):
    """Sums in float32 in any order: (terms + 2) roundings of the terms' absolute sum, then one rounding to the type (the weight's sum
    goes over ranges of tokens, which adds no more than that).  What lies behind the last row stays as it was."""
    g = torch.Generator().manual_seed(n + d + e)
    idx = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)])
    idx[torch.rand(n, k, generator=g) < 0.1] = -1
    gs, x, w = (torch.randn(*s, generator=g).to(dtype) for s in ((n, k), (n, d), (e, d)))
    idxd, gd, xd, wd = (t.to(device) for t in (idx, gs, x, w))
    s2r = torch.randperm(n * k, generator=g)
    s2r[idx.flatten() < 0] = -1
    rows = torch.randn(n * k, d, generator=g).to(dtype)

    def near(got, want, mag, terms):
        got, want, mag = got.double().cpu(), want, mag
        bound = (terms + 2) * 2.0 ** -23 * mag
        assert ((got - want).abs() <= bound * 2 + STEP[dtype] * want.abs() + 2.0 ** -24).all()   # (the last: denormal halves)

    dense = torch.zeros(n, e, dtype=torch.float64)
    for j in range(k):
        sel = idx[:, j] >= 0
        dense[sel.nonzero()[:, 0], idx[sel, j]] = gs[sel, j].double()
    grad_w, grad_b = fmoe_native.gate_weight_grad(gd, idxd, xd, e, True, any_grid=True)
    near(grad_w, dense.t() @ x.double(), dense.abs().t() @ x.double().abs(), n)
    near(grad_b, dense.sum(0), dense.abs().sum(0), n)
    part, mag = dense @ w.double(), dense.abs() @ w.double().abs()
    near(fmoe_native.reduce_slots_gate(None, None, gd, idxd, wd, any_grid=True), part, mag, k)
    picked = torch.where(s2r[:, None] >= 0, rows.double()[s2r.clamp(min=0)], torch.zeros(1, dtype=torch.float64)).view(n, k, d)
    near(fmoe_native.reduce_slots_gate(rows.to(device), s2r.to(device), gd, idxd, wd, any_grid=True), part + picked.sum(1),
         mag + picked.abs().sum(1), 2 * k)


def test_the_entry_points_for_whole_chunks_still_refuse(device):
    x = torch.randn(8, 12, device=device).to(torch.bfloat16)
    idx = torch.zeros(8, 1, dtype=torch.int64, device=device)
    with pytest.raises(Exception):
        fmoe_native.gate_weight_grad(x[:, :1].contiguous(), idx, x, 4, False)
    with pytest.raises(Exception):
        fmoe_native.reduce_slots_gate(None, None, x[:, :1].contiguous(), idx, x, any_grid=False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,d,k", [(70, 64, 3), (9, 1024, 5), (4200, 1024, 3), (4200, 1032, 7)])
def test_sums_over_an_odd_number_of_slots(n, d, k, dtype, device):
    """Slots are taken two (float32: four, eight) at a time: what is left at the end, dropped slots among them, with one and with several
    pieces of a row per wave.  float32 sums of 2 k terms, then one rounding."""
    g = torch.Generator(device=device).manual_seed(n + k)
    e = 9
    idx = torch.randn(n, e, device=device, generator=g).topk(k).indices
    idx[::7, k - 1] = -1
    rows = torch.randn(n * k, d, device=device, generator=g).to(dtype)
    w, grad = torch.randn(e, d, device=device, generator=g).to(dtype), torch.randn(n, k, device=device, generator=g).to(dtype)
    s2r = fmoe_native.route(idx, e)[2].view(-1)
    got = fmoe_native.reduce_slots_gate(rows, s2r, grad, idx, w)
    live = (idx >= 0).unsqueeze(-1)
    picked = torch.where(live, rows.double()[s2r.clamp(min=0)].view(n, k, d), 0.0)
    part = torch.where(live, w.double()[idx.clamp(min=0)] * grad.double().unsqueeze(-1), 0.0)
    want, mag = picked.sum(1) + part.sum(1), picked.abs().sum(1) + part.abs().sum(1)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    assert ((got.double() - want).abs() <= (2 * k + 1) * 2.0 ** -24 * mag + ulp * want.abs() + 2.0 ** -24).all()
