"""GPU parity of the segment table built on the device and of the grouped GEMMs launched over it
(no expert counts on the host).

The table is integer work: bit-exact against oracle.routing.segment_table.  The products over the
table run the same kernels as the host-count entry points, so with the tile shape forced they must
equal them bit for bit; beside that they are held to the float64 oracle like every other product
(1e-5 for float32, 2e-2 for bfloat16 / float16, relative to the largest reference magnitude)."""
import numpy as np
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native
from oracle import moe as omoe
from oracle import routing as orouting
from helpers import TOL, ragged_counts, rel_err, zipf_experts

pytestmark = pytest.mark.gpu

HEADER = 8


def _unpack(table, n_expert):
    """The parts of the device table that the kernels read, as numpy arrays."""
    t = table.cpu().numpy()
    seg = t[HEADER:HEADER + n_expert + 1]
    n256, n128, off256, off128 = int(t[2]), int(t[3]), int(t[4]), int(t[5])
    assert off256 % 4 == 0 and off128 % 4 == 0
    return {"n_expert": int(t[0]), "rows": int(t[1]), "seg": seg,
            "tiles256": t[off256:off256 + 4 * n256].reshape(-1, 4),
            "tiles128": t[off128:off128 + 4 * n128].reshape(-1, 4)}


def _check_table(counts, rows_cap, device):
    counts = torch.as_tensor(counts, dtype=torch.int64)
    got = _unpack(fmoe_native.segment_table(counts.to(device), rows_cap), counts.numel())
    ref = orouting.segment_table(counts.numpy(), rows_cap)
    assert got["n_expert"] == counts.numel()
    assert got["rows"] == int(ref["seg"][-1])
    assert np.array_equal(got["seg"], ref["seg"])
    for key in ("tiles256", "tiles128"):
        assert np.array_equal(got[key][:, :3], ref[key]), key
        assert not got[key][:, 3].any()


CONFIG_COUNTS = {
    "config1": lambda g: torch.bincount(torch.randint(0, 8, (8192,), generator=g), minlength=8),
    "config2": lambda g: torch.bincount(torch.randint(0, 16, (32768,), generator=g), minlength=16).clamp(max=2458),
    "config3": lambda g: torch.bincount(zipf_experts(16384, 64, 1.2, g), minlength=64),
    "config4": lambda g: torch.bincount(torch.randint(0, 8, (65536,), generator=g), minlength=8),
    "config5": lambda g: torch.bincount(torch.randint(0, 256, (65536,), generator=g), minlength=256),
}
CONFIG_SLOTS = {"config1": 8192, "config2": 32768, "config3": 16384, "config4": 65536, "config5": 65536}


@pytest.mark.parametrize("n_expert", [1, 3, 64, 512, 513, 1025])
@pytest.mark.parametrize("n_slots", [1, 63, 1024, 1025, 8192, 8193, 20000])
def test_route_with_its_segment_table(n_slots, n_expert, device):
    """Counts, positions, their inverse and the segment table of one call, on both sides of the limits of
    the one-workgroup kernel (8192 slots, 512 experts) and of the table in LDS (1024 experts): integer
    work, exact."""
    g = torch.Generator().manual_seed(n_slots + n_expert)
    gate = torch.randint(-1, n_expert, (n_slots,), generator=g)
    cnt, pos, s2r, table = fmoe_native.route_table(gate.to(device), n_expert)
    ref_pos, ref_cnt = orouting.count_by_gate(gate.numpy(), n_expert)
    total = int(ref_cnt.sum())
    assert np.array_equal(cnt.cpu().numpy(), ref_cnt)
    assert np.array_equal(pos[:total].cpu().numpy(), ref_pos) and (pos[total:] == -1).all()
    inv = np.full(n_slots, -1, dtype=np.int64)
    inv[ref_pos] = np.arange(total)
    assert np.array_equal(s2r.cpu().numpy(), inv)
    got, ref = _unpack(table, n_expert), orouting.segment_table(ref_cnt, n_slots)
    assert np.array_equal(got["seg"], ref["seg"]) and got["rows"] == total
    for key in ("tiles256", "tiles128"):
        assert np.array_equal(got[key][:, :3], ref[key]), key


@pytest.mark.parametrize("n_expert", [1, 2, 63, 64, 65])
@pytest.mark.parametrize("n_slots", [1, 64, 65, 257, 1023, 4097, 8192])
@pytest.mark.parametrize("spread", ["even", "one", "none"])
def test_table_of_the_routing_against_the_one_of_its_counts(n_slots, n_expert, spread, device):
    """The table that comes with the routing of few slots, on both sides of one expert per lane, is word for word the one that its
    own kernel builds of the counts: header, prefixes, tiles and the experts by descending rows."""
    g = torch.Generator().manual_seed(n_slots * 67 + n_expert)
    gate = torch.randint(-1, n_expert, (n_slots,), generator=g)
    if spread != "even":
        gate[torch.rand(n_slots, generator=g) < 0.9] = n_expert - 1 if spread == "one" else -1
    cnt, pos, s2r, table = fmoe_native.route_table(gate.to(device), n_expert)
    ref_pos, ref_cnt = orouting.count_by_gate(gate.numpy(), n_expert)
    total = int(ref_cnt.sum())
    assert np.array_equal(cnt.cpu().numpy(), ref_cnt)
    assert np.array_equal(pos[:total].cpu().numpy(), ref_pos) and (pos[total:] == -1).all()
    inv = np.full(n_slots, -1, dtype=np.int64)
    inv[ref_pos] = np.arange(total)
    assert np.array_equal(s2r.cpu().numpy(), inv)
    got, want = table.cpu().numpy(), fmoe_native.segment_table(cnt, n_slots).cpu().numpy()
    assert got.size == want.size
    head = HEADER + 3 * (n_expert + 1)
    assert np.array_equal(got[:head], want[:head])
    assert np.array_equal(got[-4 * n_expert:], want[-4 * n_expert:])
    for key in ("tiles256", "tiles128"):
        assert np.array_equal(_unpack(table, n_expert)[key], _unpack(torch.from_numpy(want), n_expert)[key]), key


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_tokens", [1, 7, 15, 16, 17])
@pytest.mark.parametrize("n_expert,top_k", [(1, 1), (8, 8), (33, 2), (64, 4), (64, 8)])
def test_gate_that_routes_its_own_tokens(n_tokens, n_expert, top_k, dtype, device):
    """A gate with one workgroup's tokens routes them in the same launch: routing and table of its choices, word for word those
    of the routing kernels."""
    g = torch.Generator().manual_seed(n_tokens * 65 + n_expert)
    x, w = torch.randn(n_tokens, 264, generator=g).to(dtype), torch.randn(n_expert, 264, generator=g).to(dtype)
    idx, _score, *got = fmoe_native.gate_linear_topk_route(x.to(device), w.to(device), None, top_k, 0, with_table=True)
    ref_pos, ref_cnt = orouting.count_by_gate(idx.cpu().numpy(), n_expert)
    assert np.array_equal(got[0].cpu().numpy(), ref_cnt) and np.array_equal(got[1].cpu().numpy(), ref_pos)
    want = fmoe_native.route_table(idx, n_expert)
    assert all(torch.equal(a, b) for a, b in zip(got[:3], want[:3]))
    got, want = got[3].cpu().numpy(), want[3].cpu().numpy()
    assert got.size == want.size
    head = HEADER + 3 * (n_expert + 1)
    assert np.array_equal(got[:head], want[:head]) and np.array_equal(got[-4 * n_expert:], want[-4 * n_expert:])
    for key in ("tiles256", "tiles128"):
        assert np.array_equal(_unpack(torch.from_numpy(got), n_expert)[key], _unpack(torch.from_numpy(want), n_expert)[key]), key


@pytest.mark.parametrize("name", sorted(CONFIG_COUNTS))
def test_segment_table_at_the_configurations(name, device):
    g = torch.Generator().manual_seed(11)
    _check_table(CONFIG_COUNTS[name](g), CONFIG_SLOTS[name], device)


@pytest.mark.parametrize("counts,cap", [
    ([0, 0, 0, 0], 64),                 # nothing routed at all
    ([0, 0, 0, 0], 0),                  # no slots at all
    ([5000], 5000),                     # a single expert owns every row
    ([0, 1, 0, 255, 256, 257, 0], 769), # tile edges
    ([128] * 7, 896),                   # every expert exactly one 128-row tile
    ([300, 300, 300], 700),             # counts beyond rows_cap are clamped in order
    ([-4, 10, 2 ** 40, 7], 100),        # garbage counts never overrun the tile maps
])
def test_segment_table_edge_cases(counts, cap, device):
    _check_table(counts, cap, device)


@pytest.mark.parametrize("n_expert", [1023, 1024, 1025, 4100, 8192])
def test_segment_table_many_experts(n_expert, device):
    """More experts than the kernel's 1024 threads: several passes with carried sums."""
    g = torch.Generator().manual_seed(n_expert)
    counts = torch.randint(0, 40, (n_expert,), generator=g)
    counts[torch.randperm(n_expert, generator=g)[: n_expert // 3]] = 0
    counts[n_expert // 2] = 700
    _check_table(counts, int(counts.sum()) + 17, device)


def test_segment_table_argument_checks(device):
    cnt = torch.zeros(4, dtype=torch.int64, device=device)
    small = torch.empty(4, dtype=torch.int32, device=device)
    lib = _lib.load()
    rc = lib.fmoe_segment_table_build(cnt.data_ptr(), 4, 1000, small.data_ptr(), small.numel() * 4, None)
    assert rc == -4 and b"needs" in lib.fmoe_last_error()
    assert lib.fmoe_segment_table_build(None, 4, 1000, small.data_ptr(), 1 << 20, None) == -1
    assert lib.fmoe_segment_table_bytes(-1, 4) == 0 and lib.fmoe_segment_table_bytes(10, 0) == 0
    assert lib.fmoe_linear_dev_supported(64, 128, _lib.BF16) == 1
    assert lib.fmoe_linear_dev_supported(12, 20, _lib.BF16) == 0     # rows that are not whole 16-byte chunks
    assert lib.fmoe_linear_dev_supported(64, 128, _lib.F64) == 0


TILES = ["256x256", "128x256", "128x128"]
DEV_CASES = [  # rows, slots (rows_cap), experts, in, out, empties
    (1000, 1000, 4, 64, 128, 1),
    (777, 900, 8, 256, 72, 2),        # fewer rows than slots (dropped slots): rows past the routed ones untouched
    (2048, 2048, 2, 512, 512, 0),
    (300, 300, 16, 40, 24, 5),
    (5, 64, 3, 8, 8, 1),
    (0, 32, 3, 16, 16, 3),            # no rows at all
    (1100, 1100, 2, 328, 272, 0),
    (3000, 3000, 300, 64, 96, 40),    # more experts than a host-count launch carries in its arguments
]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,slots,e,fin,fout,empties", DEV_CASES)
def test_products_over_the_device_table(dtype, rows, slots, e, fin, fout, empties, tile, device, monkeypatch):
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    g = torch.Generator().manual_seed(rows + e + fin)
    counts = ragged_counts(rows, e, g, empties) if rows else torch.zeros(e, dtype=torch.int64)
    x = torch.randn(slots, fin, generator=g).to(dtype)
    w = (torch.randn(e, fout, fin, generator=g) / fin ** 0.5).to(dtype)
    b = torch.randn(e, fout, generator=g).to(dtype)
    gy = torch.randn(slots, fout, generator=g).to(dtype)
    xd, wd, bd, gyd = x.to(device), w.to(device), b.to(device), gy.to(device)
    table = fmoe_native.segment_table(counts.to(device), slots)

    # against the host-count entry points (same kernels, same tile shape): bit for bit on the routed rows
    y, pre = fmoe_native.linear_forward_dev(xd, wd, bd, table, slots)
    assert pre is None and y.shape == (slots, fout)
    y_host = fmoe_native.linear_forward(xd, counts, wd, bd)
    assert torch.equal(y[:rows], y_host[:rows])
    gx = fmoe_native.linear_dgrad_dev(gyd, wd, table, slots)
    gw, gb = fmoe_native.linear_wgrad_dev(gyd, xd, wd, table, slots, True)
    gx_host, gw_host, gb_host = fmoe_native.linear_backward(gyd, xd, counts, wd, bd)
    assert torch.equal(gx[:rows], gx_host[:rows])
    assert torch.equal(gw, gw_host) and torch.equal(gb, gb_host)

    # against the float64 oracle
    x64, w64, b64 = x[:rows].double().requires_grad_(True), w.double().requires_grad_(True), b.double().requires_grad_(True)
    ref = omoe.per_expert_linear(x64, counts, w64, b64)
    ref.backward(gy[:rows].double())
    tol = TOL[dtype]
    assert rel_err(y[:rows], ref) <= tol
    assert rel_err(gx[:rows], x64.grad) <= tol
    assert rel_err(gw, w64.grad) <= tol and rel_err(gb, b64.grad) <= tol
    for ex in range(e):
        if counts[ex] == 0:
            assert torch.count_nonzero(gw[ex]) == 0 and torch.count_nonzero(gb[ex]) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("act", ["gelu", "relu", "none"])
def test_activation_epilogues_over_the_device_table(dtype, act, device):
    """bias + activation in the forward epilogue (with the pre-activation kept) and x act' in the data
    gradient's, rows gathered through an index in the loader: equal to the host-count entry points
    on the scattered copy, bit for bit."""
    code = {"gelu": _lib.ACT_GELU, "relu": _lib.ACT_RELU, "none": _lib.ACT_NONE}[act]
    g = torch.Generator().manual_seed(5)
    n_tokens, k, e, d, h = 700, 2, 6, 64, 192
    gate = torch.randint(-1, e, (n_tokens, k), generator=g).to(device)
    counts, pos_buf, s2r = fmoe_native.route(gate, e)
    slots = n_tokens * k
    rows = int(counts.sum())
    table = fmoe_native.segment_table(counts, slots)
    inp = torch.randn(n_tokens, d, generator=g).to(dtype).to(device)
    w = (torch.randn(e, h, d, generator=g) / d ** 0.5).to(dtype).to(device)
    b = torch.randn(e, h, generator=g).to(dtype).to(device)
    y, pre = fmoe_native.linear_forward_dev(inp, w, b, table, slots, code, True, row_index=pos_buf, index_div=k)
    scattered = fmoe_native.gather_rows(inp, pos_buf[:rows], index_div=k)
    y_host, pre_host = fmoe_native.linear_act_forward(scattered, counts.cpu(), w, b, code, True)
    assert torch.equal(y[:rows], y_host) and torch.equal(pre[:rows], pre_host)
    # data gradient of a following linear [e, d, h] with the derivative in the epilogue
    w2 = (torch.randn(e, d, h, generator=g) / h ** 0.5).to(dtype).to(device)
    gy = torch.randn(slots, d, generator=g).to(dtype).to(device)
    gx = fmoe_native.linear_dgrad_dev(gy, w2, table, slots, pre, code)
    gx_host = fmoe_native.linear_dact_backward(gy[:rows].contiguous(), counts.cpu(), w2, pre_host, code)
    assert torch.equal(gx[:rows], gx_host)


def test_unsupported_shapes_are_refused(device):
    counts = torch.tensor([3, 5], dtype=torch.int64, device=device)
    table = fmoe_native.segment_table(counts, 8)
    x = torch.randn(8, 10, device=device)        # rows of 40 bytes: not whole 16-byte chunks
    w = torch.randn(2, 20, 10, device=device)
    with pytest.raises(_lib.FmoeHipError):
        fmoe_native.linear_forward_dev(x, w, None, table, 8)
    with pytest.raises(ValueError):
        fmoe_native.linear_forward_dev(x[:4].contiguous(), w, None, table, 8)   # fewer rows than rows_cap
    with pytest.raises(ValueError):
        fmoe_native.linear_forward_dev(x, w, None, table[:10].contiguous(), 8)  # table too short


@pytest.mark.parametrize("tile", ["256x256", "128x256"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,slots,e,fin,fout", [
    (600, 700, 2, 4096, 520),     # forward: a short last round of deep tiles -> split along the contraction
    (600, 600, 3, 520, 4096),     # data gradient: the same
    (70000, 70000, 4, 3584, 264), # more than one round of tiles before the split tail
])
def test_split_tail_over_the_device_table(dtype, rows, slots, e, fin, fout, tile, device, monkeypatch):
    """A last, partial round of tiles is split along the contraction by the workgroups themselves when the
    segments come from a device table (the host does not know the tile count): same plan, same order of
    the partial sums and so the same bits as the host-count launch, with and without the caller's workspace
    (FMOE_DEV_SPLIT=0: no workspace, no split -- another order of the sums, equal within the tolerance)."""
    monkeypatch.setenv("FMOE_GEMM_TILE", tile)
    g = torch.Generator().manual_seed(rows + fin)
    counts = ragged_counts(rows, e, g, 0)
    x = torch.randn(slots, fin, generator=g).to(dtype).to(device)
    w = (torch.randn(e, fout, fin, generator=g) / fin ** 0.5).to(dtype).to(device)
    b = torch.randn(e, fout, generator=g).to(dtype).to(device)
    gy = torch.randn(slots, fout, generator=g).to(dtype).to(device)
    table = fmoe_native.segment_table(counts.to(device), slots)
    y_host = fmoe_native.linear_forward(x, counts, w, b)
    gx_host = fmoe_native.linear_backward(gy, x, counts, w, b)[0]
    for flag in ("1", "0"):
        monkeypatch.setenv("FMOE_DEV_SPLIT", flag)
        y, _ = fmoe_native.linear_forward_dev(x, w, b, table, slots)
        gx = fmoe_native.linear_dgrad_dev(gy, w, table, slots)
        if flag == "1":
            assert torch.equal(y[:rows], y_host[:rows]) and torch.equal(gx[:rows], gx_host[:rows])
        else:
            assert rel_err(y[:rows], y_host[:rows]) <= TOL[dtype] and rel_err(gx[:rows], gx_host[:rows]) <= TOL[dtype]


# counts at the edges of the 256-row tiles and of the 64-row wave tiles, experts without rows, and a last partial round of
# tiles; sizes that give the persistent kernel of the 16-bit types enough tiles for each of the three products
RING_CASES = [  # counts, in, out
    ([1, 64, 65, 127, 0, 128, 129, 255, 256, 257, 0, 511, 3000, 700, 900, 1800], 328, 4104),   # contraction and column remainders
    ([1500, 0, 2700, 3000, 1000], 3336, 4608),   # 53 slabs, 8 or 9 whole rounds and a short tail
    ([2300, 1900, 0, 3992], 8, 5000),            # one slab of one 16-byte chunk
    ([9000, 300], 4096, 4096),                   # an exact number of slabs; a tail cut along the contraction
    ([0] * 40 + [2, 1] * 30 + [700] * 12, 520, 1040),
    ([(37 * i) % 211 for i in range(1100)], 264, 520),   # more experts than the table sorts
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(RING_CASES)))
def test_persistent_kernel_products(case, dtype, device):
    """The products of many 256 x 256 tiles (one persistent workgroup per compute unit): every epilogue against
    float32 products of the same operands.  Bound per element: one rounding of the result to the element type
    (2^-8 for bfloat16, 2^-11 for float16, relative) plus 1e-3 of the rms, which covers the float32 sums in another
    order (K 2^-24 < 3e-4) and the GELU polynomials (1.4e-4)."""
    counts, fin, fout = RING_CASES[case]
    counts = torch.tensor(counts, dtype=torch.int64)
    e, rows = counts.numel(), int(counts.sum())
    slots = rows + 5
    g = torch.Generator(device=device).manual_seed(case)
    rnd = lambda *s: torch.randn(*s, device=device, generator=g)
    x, gy = rnd(slots, fin).to(dtype), rnd(slots, fout).to(dtype)
    w, b = (rnd(e, fout, fin) / fin ** 0.5).to(dtype), rnd(e, fout).to(dtype)
    pre_in = (2 * rnd(slots, fin)).to(dtype)
    table = fmoe_native.segment_table(counts.to(device), slots)
    y, pre = fmoe_native.linear_forward_dev(x, w, b, table, slots, _lib.ACT_GELU, True)
    y_np, none = fmoe_native.linear_forward_dev(x, w, b, table, slots, _lib.ACT_GELU, False)
    y_relu, _ = fmoe_native.linear_forward_dev(x, w, b, table, slots, _lib.ACT_RELU, False)
    y_plain, _ = fmoe_native.linear_forward_dev(x, w, None, table, slots)
    gx = fmoe_native.linear_dgrad_dev(gy, w, table, slots)
    gx_gelu = fmoe_native.linear_dgrad_dev(gy, w, table, slots, pre_in, _lib.ACT_GELU)
    gx_relu = fmoe_native.linear_dgrad_dev(gy, w, table, slots, pre_in, _lib.ACT_RELU)
    gw, gb = fmoe_native.linear_wgrad_dev(gy, x, w, table, slots, True)
    gw_nb, none_b = fmoe_native.linear_wgrad_dev(gy, x, w, table, slots, False)
    assert none is None and none_b is None and torch.equal(y[:rows], y_np[:rows]) and torch.equal(gw, gw_nb)

    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    def close(got, ref, what):
        bound = eps * ref.abs() + 1e-3 * ref.pow(2).mean().sqrt().clamp(min=1e-3)
        assert bool(((got.float() - ref).abs() <= bound).all()), what
    lo = 0
    for ex, n in enumerate(counts.tolist()):
        r = slice(lo, lo + n)
        lo += n
        if n == 0:
            assert torch.count_nonzero(gw[ex]) == 0 and torch.count_nonzero(gb[ex]) == 0
            continue
        xs, gs, ws, ps = x[r].float(), gy[r].float(), w[ex].float(), pre_in[r].float()
        plain = xs @ ws.t()
        full = plain + b[ex].float()
        close(y_plain[r], plain, f"expert {ex}: forward")
        close(pre[r], full, f"expert {ex}: pre-activation")
        close(y[r], torch.nn.functional.gelu(full), f"expert {ex}: gelu")
        close(y_relu[r], torch.relu(full), f"expert {ex}: relu")
        back = gs @ ws
        close(gx[r], back, f"expert {ex}: data gradient")
        ps = ps.requires_grad_(True)
        torch.nn.functional.gelu(ps).sum().backward()
        close(gx_gelu[r], back * ps.grad, f"expert {ex}: gelu derivative")
        close(gx_relu[r], back * (ps > 0), f"expert {ex}: relu derivative")
        close(gw[ex], gs.t() @ xs, f"expert {ex}: weight gradient")
        close(gb[ex], gs.sum(dim=0), f"expert {ex}: bias gradient")


FEW_ROWS = [  # counts, contraction, columns: one to four blocks of 16 rows and more than 64 rows for an expert; contractions
    # of one chunk, off the 32 elements of a product and the 128 of a unit, and of several units per wave
    ([1], 8, 8),
    ([2, 0, 1, 0, 0], 40, 24),
    ([16, 0, 0, 17, 1, 15, 0], 136, 72),
    ([33, 0, 0, 0, 0, 0], 96, 40),
    ([0, 64, 0, 1, 0, 0, 0, 0, 0, 3], 1032, 264),
    ([130, 0, 65, 0, 1] + [0] * 40, 520, 48),
    ([1, 3] * 20, 2056, 136),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(FEW_ROWS)))
def test_few_rows_per_expert(case, dtype, device):
    """The forward product of decoding steps, over sorted rows and over rows read through an index (some of whose slots
    are dropped), against the float64 oracle with the suite's tolerance of 16-bit types."""
    counts, fin, fout = FEW_ROWS[case]
    g = torch.Generator().manual_seed(case)
    cnt, e, rows, k = torch.tensor(counts), len(counts), sum(counts), 3
    slots = min(rows + 2, 8 * e)
    table = fmoe_native.segment_table(cnt.to(device), slots)
    tokens = torch.randn(rows, fin, generator=g).to(dtype)
    w = (torch.randn(e, fout, fin, generator=g) / fin ** 0.5).to(dtype)
    b = torch.randn(e, fout, generator=g).to(dtype)
    index = torch.full((slots,), -1, dtype=torch.int64)
    index[:rows] = torch.randint(0, rows * k, (rows,), generator=g)
    tol = TOL[dtype]
    for row_index in (None, index):
        x = tokens if row_index is None else tokens[row_index[:rows] // k]
        ref = omoe.per_expert_linear(x.double(), cnt, w.double(), b.double())
        xd = tokens if row_index is not None else torch.cat([tokens, tokens.new_zeros(slots - rows, fin)])
        args = dict(row_index=None if row_index is None else row_index.to(device), index_div=1 if row_index is None else k)
        y, pre = fmoe_native.linear_forward_dev(xd.to(device), w.to(device), b.to(device), table, slots, _lib.ACT_GELU, True, **args)
        assert rel_err(pre[:rows], ref) <= tol and rel_err(y[:rows], torch.nn.functional.gelu(ref)) <= tol
        y, none = fmoe_native.linear_forward_dev(xd.to(device), w.to(device), b.to(device), table, slots, _lib.ACT_RELU, False, **args)
        assert none is None and rel_err(y[:rows], ref.relu()) <= tol
        y, _ = fmoe_native.linear_forward_dev(xd.to(device), w.to(device), None, table, slots, **args)
        assert rel_err(y[:rows], omoe.per_expert_linear(x.double(), cnt, w.double(), None)) <= tol


@pytest.mark.parametrize("fin,fout", [(4, 8), (60, 68), (64, 132), (100, 260)])
@pytest.mark.parametrize("counts", [[1], [63, 0, 64, 65], [127, 128, 129, 0], [192, 193, 1], [300, 0, 5]])
def test_float32_tiles_of_64(counts, fin, fout, device, monkeypatch):
    """float32 in 64 x 64 tiles, which take the halves of the table's 128-row tiles: every product over the device table
    and over host counts, the same bits from both, against the float64 oracle."""
    monkeypatch.setenv("FMOE_GEMM_TILE", "64x64")
    g = torch.Generator().manual_seed(sum(counts) + fin)
    cnt, e, rows = torch.tensor(counts), len(counts), sum(counts)
    table = fmoe_native.segment_table(cnt.to(device), rows)
    x, gy = torch.randn(rows, fin, generator=g), torch.randn(rows, fout, generator=g)
    w, b = torch.randn(e, fout, fin, generator=g) / fin ** 0.5, torch.randn(e, fout, generator=g)
    pre_in = torch.randn(rows, fin, generator=g)
    x64, w64, b64 = (t.double().requires_grad_(True) for t in (x, w, b))
    ref = omoe.per_expert_linear(x64, cnt, w64, b64)
    ref.backward(gy.double())
    xd, wd, bd, gyd, pd = (t.to(device) for t in (x, w, b, gy, pre_in))
    y, pre = fmoe_native.linear_forward_dev(xd, wd, bd, table, rows, _lib.ACT_GELU, True)
    y_h, pre_h = fmoe_native.linear_act_forward(xd, cnt, wd, bd, _lib.ACT_GELU)
    gx = fmoe_native.linear_dgrad_dev(gyd, wd, table, rows)
    gx_act = fmoe_native.linear_dgrad_dev(gyd, wd, table, rows, pd, _lib.ACT_RELU)
    gw, gb = fmoe_native.linear_wgrad_dev(gyd, xd, wd, table, rows, True)
    gx_h, gw_h, gb_h = fmoe_native.linear_backward(gyd, xd, cnt, wd, bd)
    for got, host in ((y, y_h), (pre, pre_h), (gx, gx_h), (gw, gw_h), (gb, gb_h)):
        assert torch.equal(got, host)
    tol = TOL[torch.float32]
    assert rel_err(pre, ref) <= tol and rel_err(y, torch.nn.functional.gelu(ref)) <= tol
    assert rel_err(gx, x64.grad) <= tol and rel_err(gx_act, x64.grad * (pre_in > 0)) <= tol
    assert rel_err(gw, w64.grad) <= tol and rel_err(gb, b64.grad) <= tol


@pytest.mark.parametrize("n_expert", [1, 2, 63, 64, 65, 255, 256, 257, 300, 512, 513, 1023, 1024, 1025, 1300])
@pytest.mark.parametrize("kind", ["random", "equal", "few", "ascending"])
def test_order_of_the_experts_by_their_rows(n_expert, kind, device):
    """The table's list of {expert, first row, rows} in descending order of the rows, of equal ones the lower expert first;
    beyond 1024 experts in expert order.  From the stand-alone table and from the one of a routing call: exact."""
    g = torch.Generator().manual_seed(n_expert)
    counts = {"random": torch.randint(0, 40, (n_expert,), generator=g), "equal": torch.full((n_expert,), 3),
              "few": (torch.rand(n_expert, generator=g) < 0.05).long() * 7, "ascending": torch.arange(n_expert) % 50}[kind]
    gate = torch.repeat_interleave(torch.arange(n_expert), counts)
    gate = gate[torch.randperm(gate.numel(), generator=g)]
    slots = gate.numel() + 1
    gate = torch.cat([gate, torch.tensor([-1])])
    first = np.concatenate([[0], np.cumsum(counts.numpy())[:-1]])
    experts = sorted(range(n_expert), key=lambda e: (-int(counts[e]), e)) if n_expert <= 1024 else list(range(n_expert))
    want = [(e, int(first[e]), int(counts[e]), 0) for e in experts]
    for table in (fmoe_native.segment_table(counts.to(device), slots), fmoe_native.route_table(gate.to(device), n_expert)[3]):
        t = table.cpu().numpy()
        # (behind the map of the 128-row tiles, laid out for the most there can be)
        at = int(t[5]) + 4 * (slots // 128 + min(n_expert, slots))
        assert [tuple(r) for r in t[at:at + 4 * n_expert].reshape(-1, 4).tolist()] == want


@pytest.mark.parametrize("rows_cap", [(1 << 22) - 1, 1 << 22, 1 << 23])
@pytest.mark.parametrize("n_expert", [193, 700, 1024])
def test_order_of_experts_with_many_rows(n_expert, rows_cap, device):
    """The same list on either side of the number of rows that sorts by 32-bit keys; one expert with nearly all rows."""
    g = torch.Generator().manual_seed(n_expert)
    counts = torch.randint(0, 3, (n_expert,), generator=g)
    counts[n_expert // 2] = rows_cap - int(counts.sum()) + int(counts[n_expert // 2])
    t = fmoe_native.segment_table(counts.to(device), rows_cap).cpu().numpy()
    first = np.concatenate([[0], np.cumsum(counts.numpy())[:-1]])
    want = [(e, int(first[e]), int(counts[e]), 0) for e in sorted(range(n_expert), key=lambda e: (-int(counts[e]), e))]
    at = int(t[5]) + 4 * (rows_cap // 128 + n_expert)
    assert [tuple(r) for r in t[at:at + 4 * n_expert].reshape(-1, 4).tolist()] == want


UNEVEN = [  # experts, in, out, rows, routing: weight gradients whose tiles are dealt by cost, and some on either side of that rule
    (64, 1456, 1256, 12926, "zipf"),
    (32, 544, 8040, 3000, "one"),
    (512, 264, 512, 9000, "few"),
    (1024, 520, 256, 20000, "zipf"),
    (1030, 256, 264, 5000, "zipf"),       # (more experts than the plan takes)
    (8, 2600, 2600, 20000, "zipf"),
    (16, 1296, 1800, 700, "one"),
    (513, 256, 256, 30000, "one"),        # one tile per expert
    (9, 2048, 2048, 3000, "even"),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("e,fin,fout,rows,routing", UNEVEN)
def test_weight_gradient_of_uneven_experts(e, fin, fout, rows, routing, dtype, device):
    """Every tile of the weight gradient is computed once, however the tiles are dealt to the persistent workgroups: into memory
    that held NaN before, against float32 products, with the bound of the persistent kernel's other products."""
    g = torch.Generator().manual_seed(e + rows)
    p = {"zipf": torch.arange(1, e + 1).float() ** -1.2, "one": (torch.arange(e) == e // 3).float(),
         "few": (torch.arange(e) % 37 == 5).float(), "even": torch.ones(e)}[routing]
    counts = torch.bincount(torch.multinomial(p[torch.randperm(e, generator=g)], rows, replacement=True, generator=g), minlength=e)
    slots = rows + 3
    gd = torch.Generator(device=device).manual_seed(e)
    x = torch.randn(slots, fin, device=device, generator=gd).to(dtype)
    gy = torch.randn(slots, fout, device=device, generator=gd).to(dtype)
    weight = torch.empty(e, fout, fin, dtype=dtype, device=device)
    table = fmoe_native.segment_table(counts.to(device), slots)
    for size in ((e, fout, fin), (e, fout)):
        torch.full(size, float("nan"), dtype=dtype, device=device)   # (freed at once: the next tensor of this size takes its place)
    gw, gb = fmoe_native.linear_wgrad_dev(gy, x, weight, table, slots, True)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    lo = 0
    for ex, n in enumerate(counts.tolist()):
        gs, xs = gy[lo:lo + n].float(), x[lo:lo + n].float()
        lo += n
        for got, ref in ((gw[ex], gs.t() @ xs), (gb[ex], gs.sum(dim=0))):
            bound = eps * ref.abs() + 1e-3 * ref.pow(2).mean().sqrt() if n else torch.zeros_like(ref)
            assert bool(((got.float() - ref).abs() <= bound).all()), f"expert {ex} with {n} rows"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,fin,fout", [
    ([0] * 600, 264, 520),                                        # no expert has rows
    ([0] * 127 + [5], 96, 3264),
    ([3] + [0] * 15 + [200] + [0] * 15, 1288, 1000),
    ([0, 1] * 300, 8, 2056),                                      # gradients of one piece and a little
    ([0] * 9 + [300] + [0] * 70, 2048, 1032),                     # whole pieces
    ([0] * 1000 + [2] * 24, 256, 256),
    ([0] * 1029 + [2], 256, 264),                                 # more experts than the table sorts
])
def test_weight_gradient_of_experts_without_rows(counts, fin, fout, dtype, device):
    """Large launches fill the gradients of experts without rows apart from the products' tiles: exact zeros there, in memory
    that held NaN before, and the float32 products, rounded, for the others; the table's count of experts with rows."""
    counts = torch.tensor(counts)
    e, slots = counts.numel(), int(counts.sum()) + 2
    g = torch.Generator(device=device).manual_seed(e)
    x = torch.randn(slots, fin, device=device, generator=g).to(dtype)
    gy = torch.randn(slots, fout, device=device, generator=g).to(dtype)
    weight = torch.empty(e, fout, fin, dtype=dtype, device=device)
    table = fmoe_native.segment_table(counts.to(device), slots)
    assert int(table[7]) == (int((counts > 0).sum()) if e <= 1024 else e)
    for size in ((e, fout, fin), (e, fout)):
        torch.full(size, float("nan"), dtype=dtype, device=device)   # (freed at once: the next tensor of this size takes its place)
    gw, gb = fmoe_native.linear_wgrad_dev(gy, x, weight, table, slots, True)
    empty = (counts == 0).to(device)
    assert not gw[empty].any() and not gb[empty].any()
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    first = torch.cumsum(counts, 0) - counts
    for ex in torch.nonzero(counts).flatten().tolist():
        lo, n = int(first[ex]), int(counts[ex])
        gs, xs = gy[lo:lo + n].float(), x[lo:lo + n].float()
        for got, ref in ((gw[ex], gs.t() @ xs), (gb[ex], gs.sum(dim=0))):
            assert bool(((got.float() - ref).abs() <= eps * ref.abs() + 1e-3 * ref.pow(2).mean().sqrt()).all()), f"expert {ex}"
