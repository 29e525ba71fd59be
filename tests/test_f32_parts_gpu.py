"""float32 products out of bf16 parts: each tile shape at the edges of its rows, columns and slabs, the distance from float64,
and what no sum of bf16 numbers stands for (infinities, NaN, the largest floats)."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu

TILES = ["64x64", "128x128", "128x128+"]
EDGES = [1, 0, 63, 64, 65, 127, 128, 129, 191, 300]


def operands(counts, k, n, device, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    e, rows = len(counts), sum(counts)
    x = (torch.randn(rows, k, generator=g) * scale).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(device)
    gy = torch.randn(rows, n, generator=g).to(device)
    return x, w, gy, fmoe_native.segment_table(torch.tensor(counts).to(device), rows)


def products(x, w, gy, table):
    rows = x.shape[0]
    return (fmoe_native.linear_forward_dev(x, w, None, table, rows)[0], fmoe_native.linear_dgrad_dev(gy, w, table, rows),
            *fmoe_native.linear_wgrad_dev(gy, x, w, table, rows, True))


def reference(x, w, gy, counts):
    """Float64 products and the sums of the terms' sizes."""
    x, w, gy = x.double(), w.double(), gy.double()
    ends = torch.tensor(counts).cumsum(0).tolist()
    segs = [(z - c, z) for c, z in zip(counts, ends)]
    size = lambda *t: [v.abs() for v in t]
    def all_of(x, w, gy):
        return (torch.cat([x[a:z] @ w[i].t() for i, (a, z) in enumerate(segs)]), torch.cat([gy[a:z] @ w[i] for i, (a, z) in enumerate(segs)]),
                torch.stack([gy[a:z].t() @ x[a:z] for a, z in segs]), torch.stack([gy[a:z].sum(0) for a, z in segs]))
    return all_of(x, w, gy), all_of(*size(x, w, gy))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("k,n", [(4, 4), (32, 132), (36, 60), (68, 128), (160, 264), (2052, 68)])
def test_products(k, n, tile, device, monkeypatch):
    """A contraction of K terms in any order is off by at most K roundings of 2^-24 of the terms' sizes; each term leaves out 2^-25."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    x, w, gy, table = operands(EDGES, k, n, device, k + n)
    want, sizes = reference(x, w, gy, EDGES)
    for got, ref, size, terms in zip(products(x, w, gy, table), want, sizes, (k, n, max(EDGES), max(EDGES))):
        assert ((got.double() - ref).abs() <= (terms + 2) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30])
def test_distance_from_float64(tile, scale, device, monkeypatch):
    """No further off than a float32 product whose K roundings add up like a random walk: 2^-24 sqrt(K / 3) of the root of the summed
    squares, on which the fp32 matrix instruction comes to 1.2 to 1.5 and these to 1.0 to 1.3."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    counts, k, n = [512, 512], 512, 512
    x, w, gy, table = operands(counts, k, n, device, 7, scale)
    want, _ = reference(x, w, gy, counts)
    for got, ref in zip(products(x, w, gy, table)[:3], want):
        assert (got.double() - ref).norm() <= 1.4 * 2.0 ** -24 * (512 / 3) ** 0.5 * ref.norm()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38, -3.402e38])
def test_what_bf16_does_not_hold(value, tile, device, monkeypatch):
    """The rows and columns that a large value reaches are what float64 rounded to float32 has, the others as without it."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    counts, k, n = [130, 3, 70], 132, 136
    x, w, gy, table = operands(counts, k, n, device, 11)
    gy /= 8   # (a product with the largest floats stays finite)
    x[129, 77] = value
    x[131, 3] = value
    want, sizes = reference(x, w, gy, counts)
    for got, ref, size, terms in zip(products(x, w, gy, table), want, sizes, (k, n, 130, 130)):
        ref32, size = ref.float(), size.nan_to_num(posinf=0.0)
        assert torch.equal(got.isnan(), ref32.isnan()) and torch.equal(got.isinf(), ref32.isinf())
        assert torch.equal(got[got.isinf()], ref32[got.isinf()])
        at = ref32.isfinite()
        assert ((got.double() - ref)[at].abs() <= (terms + 2) * 2.0 ** -24 * size[at]).all()


def test_an_infinite_row_in_a_tail_whose_contraction_is_shared(device, monkeypatch):
    monkeypatch.setenv("FMOE_GEMM_TILE", "128x128")
    x, w, gy, table = operands([40, 0, 7], 4100, 264, device, 13)
    x[41, 4000] = float("inf")
    got = fmoe_native.linear_forward_dev(x, w, None, table, 47)[0]
    assert torch.equal(got[41], torch.full_like(got[41], float("inf")) * w[2, :, 4000].sign())
    rest = [i for i in range(47) if i != 41]
    ref = torch.cat([x[:40].double() @ w[0].double().t(), x[40:].double() @ w[2].double().t()])
    assert (got[rest].double() - ref[rest]).abs().max() <= 4102 * 2.0 ** -24 * ref[rest].abs().max()


def test_few_and_many_rows_take_a_shape_by_themselves(device, monkeypatch):
    monkeypatch.delenv("FMOE_GEMM_TILE", raising=False)
    for counts, k, n in (([200, 0, 56], 512, 640), ([700, 1, 900, 300], 640, 1280), ([64] * 24, 576, 576)):
        x, w, gy, table = operands(counts, k, n, device, n)
        want, sizes = reference(x, w, gy, counts)
        for got, ref, size, terms in zip(products(x, w, gy, table), want, sizes, (k, n, max(counts), max(counts))):
            assert ((got.double() - ref).abs() <= (terms + 2) * 2.0 ** -24 * size).all()
        pre = fmoe_native.linear_forward_dev(x, w, None, table, sum(counts), _lib.ACT_GELU, True)[1]
        assert torch.equal(pre, fmoe_native.linear_forward_dev(x, w, None, table, sum(counts))[0])


def of_kind(kind, rows, cols, g, device):
    z = torch.randn(rows, cols, generator=g)
    return {"normal": z, "relu": z.clamp(min=0), "one sign": z.abs()}[kind].to(device)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("left,right", [("normal", "normal"), ("relu", "normal"), ("one sign", "one sign")])
def test_the_accumulator_is_rounded_by_one_product_only(left, right, tile, device, monkeypatch):
    """The largest of the six products rounds the accumulator once per 8 elements: m = K / 8 roundings of 2^-24 / sqrt(3) of what has
    been added up, sqrt(i / m) of the sum after i of them (less where all terms have one sign), come to 2^-24 sqrt(m / 6) of it.  With all six products in one
    accumulator, and on the fp32 matrix instruction, it is more than that, and the roundings of the former lie to one side: 0.09 to 0.2 of the distance."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    r, k, n = 256, 2048, 192
    g = torch.Generator().manual_seed(17)
    a, b = of_kind(left, r, k, g, device), of_kind(right, n, k, g, device)
    ref = a.double() @ b.double().t()
    rows, terms = (fmoe_native.segment_table(torch.tensor([c]).to(device), c) for c in (r, k))
    for got in (fmoe_native.linear_forward_dev(a, b.view(1, n, k), None, rows, r)[0],
                fmoe_native.linear_dgrad_dev(a, b.t().contiguous().view(1, k, n), rows, r),
                fmoe_native.linear_wgrad_dev(a.t().contiguous(), b.t().contiguous(), torch.empty(1, r, n, device=device), terms, k, False)[0][0]):
        err = got.double() - ref
        assert err.norm() <= 2.0 ** -24 * (k / 8 / 6) ** 0.5 * ref.norm()
        if right == "normal":
            assert err.mean().abs() <= err.square().mean().sqrt() / 16


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("power", [-96, -112, -120, -126])
def test_rows_of_tiny_elements(power, tile, device, monkeypatch):
    """Rows of either operand that are small throughout keep float32's digits (2^-24 sqrt(K) of the products' root of summed squares bounds the random walk
    of K roundings); the other rows, and rows of zeros, are as without them."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    counts, k, n = [130, 3, 70], 512, 136
    x, w, gy, table = operands(counts, k, n, device, 23)
    x[5] *= 2.0 ** power
    x[:, 9] *= 2.0 ** power
    x[132] = 0
    w[2, 77] *= 2.0 ** power
    gy[150:] *= 2.0 ** power
    gy[:, 3] *= 2.0 ** power
    want, _ = reference(x, w, gy, counts)
    fwd, dgrad, wgrad = zip(products(x, w, gy, table)[:3], want[:3])
    parts = {"row": [t[5] for t in fwd], "zeros": [t[132] for t in fwd], "weight": [t[133:, 77] for t in fwd], "gradient rows": [t[150:] for t in dgrad],
             "input column": [t[..., 9] for t in wgrad], "gradient column": [t[:, 3] for t in wgrad], "all": fwd, "all d": dgrad, "all w": wgrad}
    for name, (got, ref) in parts.items():
        subnormal = 2.0 ** -149 * ref.numel() ** 0.5
        assert (got.double() - ref).norm() <= 2.0 ** -24 * k ** 0.5 * ref.norm() + subnormal, name
