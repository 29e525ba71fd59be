"""Row-ragged products of the 16-bit types whose slabs are requested by waves of their own: the three tile shapes at the edges of
their rows, columns and slab counts, and what picks a shape."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native

pytestmark = pytest.mark.gpu

# a product's sums run in float32 on both sides, in another order; the result is rounded once
HALF_STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
EDGES = [1, 0, 15, 16, 63, 64, 65, 127, 128, 129, 191, 300]
CASES = [  # counts, contraction, columns
    (EDGES, 8, 8),          # one chunk of one slab
    (EDGES, 64, 136),
    (EDGES, 72, 120),       # a slab and a chunk
    (EDGES, 192, 128),      # fewer slabs than are requested ahead
    (EDGES, 320, 264),      # more
    ([40, 0, 7], 4104, 264),   # long: the tail's contraction is shared where the shape allows
]


def close(got, want, dtype, contraction):
    """One rounding to ``dtype`` plus the float32 sums of ``contraction`` terms in two orders (each term at most about 4 sigma)."""
    want = want.double()
    bound = HALF_STEP[dtype] * want.abs() + contraction ** 0.5 * 2.0 ** -22 * 16
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("tile", ["64x128", "128x128+", "128x128"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_products(case, dtype, tile, device, monkeypatch):
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    counts, k, n = CASES[case]
    e, rows = len(counts), sum(counts)
    slots = rows + 70
    g = torch.Generator().manual_seed(case)
    cnt = torch.tensor(counts)
    table = fmoe_native.segment_table(cnt.to(device), slots)
    x = torch.randn(slots, k, generator=g).to(dtype).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(dtype).to(device)
    b = torch.randn(e, n, generator=g).to(dtype).to(device)
    ends = cnt.cumsum(0).tolist()
    segs = [(end - c, end) for c, end in zip(counts, ends)]
    ref = torch.cat([x[lo:hi].double() @ w[i].double().t() + b[i].double() for i, (lo, hi) in enumerate(segs)])
    got, _ = fmoe_native.linear_forward_dev(x, w, b, table, slots)
    close(got[:rows], ref, dtype, k)
    # through an index, two slots to a token; entries that name no token read zeros
    index = torch.randint(0, 2 * slots, (slots,), generator=g)
    index[torch.rand(slots, generator=g) < 0.1] = -1
    picked = torch.where(index[:, None].to(device) >= 0, x[(index // 2).clamp(min=0).to(device)], torch.zeros_like(x))
    ref_g = torch.cat([picked[lo:hi].double() @ w[i].double().t() + b[i].double() for i, (lo, hi) in enumerate(segs)])
    got, pre = fmoe_native.linear_forward_dev(x, w, b, table, slots, _lib.ACT_RELU, True, row_index=index.to(device), index_div=2)
    close(pre[:rows], ref_g, dtype, k)
    assert torch.equal(got[:rows], pre[:rows].clamp(min=0))
    # data gradients: of the same linear, and through the activation of the one before
    gy = torch.randn(slots, n, generator=g).to(dtype).to(device)
    gx = fmoe_native.linear_dgrad_dev(gy, w, table, slots)
    ref_x = torch.cat([gy[lo:hi].double() @ w[i].double() for i, (lo, hi) in enumerate(segs)])
    close(gx[:rows], ref_x, dtype, n)
    gated = fmoe_native.linear_dgrad_dev(gy, w, table, slots, x, _lib.ACT_RELU)
    assert torch.equal(gated[:rows], torch.where(x[:rows] > 0, gx[:rows], torch.zeros_like(gx[:rows])))
    # the same launches over host counts
    assert torch.equal(fmoe_native.linear_forward(x, cnt, w, b)[:rows], fmoe_native.linear_forward_dev(x, w, b, table, slots)[0][:rows])


@pytest.mark.parametrize("counts,k,n", [([60] * 4, 512, 256), ([130, 0, 500], 256, 2048), ([200] * 12, 1024, 1024), ([600] * 8, 512, 2048),
                                        ([1100] * 6, 256, 3072), ([1] * 200, 128, 128)])
def test_the_shape_that_is_picked_changes_no_bit(counts, k, n, device, monkeypatch):
    """Every shape adds an element's products in the order of the contraction, so whichever the estimate picks -- over host counts,
    which it knows, or a device table, which it guesses -- gives what a forced one gives."""
    e, rows = len(counts), sum(counts)
    g = torch.Generator().manual_seed(rows)
    cnt = torch.tensor(counts)
    table = fmoe_native.segment_table(cnt.to(device), rows)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(e, n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(device)
    gy = torch.randn(rows, n, generator=g).to(torch.bfloat16).to(device)

    def products():
        return (fmoe_native.linear_forward(x, cnt, w), fmoe_native.linear_dgrad_dev(gy, w, table, rows),
                fmoe_native.linear_backward(gy, x, cnt, w)[0])

    monkeypatch.delenv("FMOE_GEMM_TILE", raising=False)
    picked = products()
    for tile in ("64x128", "128x128+", "128x128", "128x256", "256x256"):
        monkeypatch.setenv("FMOE_GEMM_TILE", tile)
        for a, b in zip(picked, products()):
            assert torch.equal(a, b), tile
