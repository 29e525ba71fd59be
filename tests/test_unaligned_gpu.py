"""GPU parity of the grouped GEMM for 16-bit types off the 16-byte grid (feature sizes that are no multiple of
eight, or tensors that begin at any element) against the float64 oracle.

The tolerance is the suite's for 16-bit types: one rounding of the result (2^-8 for bfloat16) and products of
rounded inputs, relative to the largest reference magnitude."""
import pytest
import torch

from fastermoe_amd import FMoETransformerMLP, _lib, fmoe_native
from oracle import moe as omoe
from helpers import TOL, rel_err

pytestmark = pytest.mark.gpu

CASES = [  # counts, in, out: edges of the 64- and 128-row tiles, of the 128 columns and of the 64-element slabs
    ([1], 1, 1),
    ([7, 0, 9], 3, 5),
    ([63, 64, 65], 63, 127),
    ([127, 128, 129, 0], 65, 129),
    ([200, 1, 30], 127, 255),
    ([64, 0, 131], 130, 68),
    ([300, 150], 257, 191),
    ([130] * 5, 500, 1302),
    ([4100, 0, 4000], 150, 1100),       # enough tiles for the 128-row ones
    ([3] * 300, 12, 20),                # more experts than one launch takes
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,fin,fout", CASES)
def test_sizes_off_the_grid(dtype, counts, fin, fout, device):
    _check(dtype, counts, fin, fout, device, 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shift", [1, 2, 5])
def test_tensors_at_any_element(dtype, shift, device):
    _check(dtype, [70, 0, 130], 192, 136, device, shift)


def _at(t, shift, device):
    """A contiguous copy of ``t`` on the device that begins ``shift`` elements past an aligned address."""
    buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=device)
    out = buf[shift:].view(t.shape)
    out.copy_(t)
    return out


def _check(dtype, counts, fin, fout, device, shift):
    g = torch.Generator().manual_seed(sum(counts) + fin + fout)
    cnt, e, rows = torch.tensor(counts), len(counts), sum(counts)
    x = torch.randn(rows, fin, generator=g).to(dtype)
    w = (torch.randn(e, fout, fin, generator=g) / fin ** 0.5).to(dtype)
    b = torch.randn(e, fout, generator=g).to(dtype)
    gy = torch.randn(rows, fout, generator=g).to(dtype)
    pre_in = torch.randn(rows, fin, generator=g).to(dtype)
    x64, w64, b64 = (t.double().requires_grad_(True) for t in (x, w, b))
    y64 = omoe.per_expert_linear(x64, cnt, w64, b64)
    y64.backward(gy.double())
    xd, wd, bd, gyd, pd = (_at(t, shift, device) for t in (x, w, b, gy, pre_in))
    tol = TOL[dtype]
    y, pre = fmoe_native.linear_act_forward(xd, cnt, wd, bd, _lib.ACT_GELU)
    assert rel_err(pre, y64) <= tol
    assert rel_err(y, torch.nn.functional.gelu(y64)) <= tol
    assert rel_err(fmoe_native.linear_forward(xd, cnt, wd, bd), y64) <= tol
    gx, gw, gb = fmoe_native.linear_backward(gyd, xd, cnt, wd, bd)
    assert rel_err(gx, x64.grad) <= tol and rel_err(gw, w64.grad) <= tol and rel_err(gb, b64.grad) <= tol
    for ex in range(e):
        if counts[ex] == 0:
            assert torch.count_nonzero(gw[ex]) == 0 and torch.count_nonzero(gb[ex]) == 0
    p64 = pre_in.double().requires_grad_(True)
    torch.nn.functional.gelu(p64).backward(x64.grad)
    assert rel_err(fmoe_native.linear_dact_backward(gyd, cnt, wd, pd, _lib.ACT_GELU), p64.grad) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,fin,fout", [([0, 3, 0, 0], 1, 1), ([0, 1, 0], 3, 5), ([0] * 40 + [2] + [0] * 9, 1483, 70),
                                             ([0, 5, 0, 0, 200], 129, 257)])
def test_weight_gradients_of_experts_without_rows(dtype, counts, fin, fout, device):
    """Zeros wherever an expert's gradient begins, into memory that held NaN before, and nothing beyond them."""
    x = torch.randn(sum(counts), fin, device=device).to(dtype)
    gy = torch.randn(sum(counts), fout, device=device).to(dtype)
    w = torch.empty(len(counts), fout, fin, dtype=dtype, device=device)
    b = torch.empty(len(counts), fout, dtype=dtype, device=device)
    for size in (w.shape, b.shape):
        torch.full(size, float("nan"), dtype=dtype, device=device)   # (freed at once: the next tensor of this size takes its place)
    gw, gb = fmoe_native.linear_weight_backward(gy, x, torch.tensor(counts), w, b)
    lo = 0
    for ex, n in enumerate(counts):
        gs, xs = gy[lo:lo + n].double(), x[lo:lo + n].double()
        lo += n
        if n:
            assert rel_err(gw[ex], gs.t() @ xs) <= TOL[dtype] and rel_err(gb[ex], gs.sum(dim=0)) <= TOL[dtype]
        else:
            assert not gw[ex].any() and not gb[ex].any()


@pytest.mark.parametrize("dtype,n,d,h,e,shift", [
    (torch.bfloat16, 4096, 4096, 4096, 4, 4),   # sizes at which a fused layer leaves its chunks where it may
    (torch.bfloat16, 300, 128, 256, 4, 1),
    (torch.float32, 300, 128, 256, 4, 1),
])
@pytest.mark.parametrize("what", ["parameters", "input"])
@pytest.mark.parametrize("fuse", [False, True])
def test_layer_over_tensors_at_any_element(dtype, n, d, h, e, shift, what, fuse, device, monkeypatch):
    """Expert weights and biases that are views into a larger buffer, or token rows that are: the same results as over
    tensors of their own, fused and unfused.  Bound: the suite's tolerance of the type, twice (two runs with
    their sums in different orders)."""
    monkeypatch.delenv("FMOE_FUSE_GRAN", raising=False)
    torch.manual_seed(shift)
    with device:
        moe = FMoETransformerMLP(num_expert=e, d_model=d, d_hidden=h, top_k=2)
    moe = moe.to(dtype)
    moe.enable_fuse = fuse
    with torch.no_grad():
        for lin in (moe.experts.htoh4, moe.experts.h4toh):
            lin.weight.normal_(0, lin.weight.shape[2] ** -0.5)
            lin.bias.normal_()
    x = torch.randn(n, d, device=device).to(dtype)
    grad = torch.randn(n, d, device=device).to(dtype)

    def step(inp):
        moe.zero_grad(set_to_none=True)
        leaf = inp.detach().requires_grad_(True)
        out = moe(leaf)
        out.backward(grad)
        return [out.detach(), leaf.grad] + [p.grad for p in moe.experts.parameters()]

    want = step(x)
    if what == "parameters":
        for p in moe.experts.parameters():
            p.data = _at(p.data, shift, device)
            assert p.data_ptr() % 16 != 0
    else:
        x = _at(x, shift, device)
        assert x.data_ptr() % 16 != 0
    for got, ref in zip(step(x), want):
        assert rel_err(got, ref) <= 2 * TOL[dtype]
