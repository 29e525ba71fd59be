"""GPU parity of the routing / capacity kernels: bit-exact against the CPU oracle
and the committed golden cases, through the operator module (which calls the C ABI)."""
import json
import os

import numpy as np
import pytest
import torch

from fastermoe_amd import fmoe_native
from fastermoe_amd.functions import count_by_gate, prepare_forward
from fastermoe_amd.gates.utils import limit_by_capacity
from oracle import routing as orouting
from helpers import TOL, rel_err

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "routing_cases.json")


def _cases():
    with open(GOLDEN) as f:
        return json.load(f)


def _dev(a, device, dtype):
    return torch.as_tensor(np.asarray(a), dtype=dtype).to(device)


@pytest.mark.parametrize("case", _cases(), ids=lambda c: c["name"])
def test_golden_cases(case, device):
    e = case["n_expert"]
    gate = _dev(case["gate"], device, torch.int64)
    cnt = torch.zeros(e, dtype=torch.int32, device=device)
    fmoe_native.expert_count(gate, cnt)
    assert cnt.cpu().tolist() == case["counts"]
    cum = torch.cumsum(cnt.long(), 0).int()
    pos = torch.full((sum(case["counts"]),), -7, dtype=torch.int64, device=device)
    fmoe_native.assign_pos(cum, gate, pos)
    assert pos.cpu().tolist() == case["pos"]
    if len(case["gate"]):
        assert cum.cpu().tolist() == case["cum_after"]
    cap = torch.full((e,), case["capacity"], dtype=torch.int32, device=device)
    lim = fmoe_native.limit_by_capacity(cnt.long(), cap, e, 1)
    assert lim.cpu().tolist() == case["limited"]
    ec = lim.int()
    pruned = fmoe_native.prune_gate_by_capacity(gate, ec, e, 1)
    assert pruned.cpu().tolist() == case["pruned"]
    if len(case["gate"]):
        assert ec.cpu().tolist() == case["cap_after"]
    # fused route
    c2, pos2, s2r = fmoe_native.route(gate, e)
    assert c2.cpu().tolist() == case["counts"]
    total = sum(case["counts"])
    assert pos2[:total].cpu().tolist() == case["pos"]
    inv = [-1] * len(case["gate"])
    for row, slot in enumerate(case["pos"]):
        inv[slot] = row
    assert s2r.cpu().tolist() == inv


SHAPES = [  # (n_tokens, top_k, n_expert, drop_fraction)
    (4096, 2, 8, 0.0),       # config 1
    (16384, 2, 16, 0.0),     # config 2
    (16384, 1, 64, 0.0),     # config 3 (Zipf below)
    (32768, 2, 8, 0.0),      # config 4
    (8192, 8, 256, 0.0),     # config 5
    (1000, 3, 7, 0.3),       # ragged sizes, dropped slots
    (2049, 1, 1, 0.0),       # one expert, one slot past a workgroup boundary
    (63, 2, 300, 0.1),       # more experts than slots
    (5000, 2, 8192, 0.0),    # largest supported expert count
]


@pytest.mark.parametrize("n,k,e,drop", SHAPES)
def test_route_bit_exact(n, k, e, drop, device):
    rng = np.random.default_rng(n + k + e)
    if e == 64:
        p = (np.arange(1, e + 1) ** -1.2)
        gate = rng.permutation(e)[rng.choice(e, size=(n, k), p=p / p.sum())]
    else:
        gate = rng.integers(0, e, size=(n, k))
    gate = gate.astype(np.int64)
    gate[rng.random((n, k)) < drop] = -1
    ref_pos, ref_cnt = orouting.count_by_gate(gate, e)
    g = torch.from_numpy(gate).to(device)
    if k == 1:
        g = g.view(-1)

    pos, lec, all_ec, gec, all_gec = count_by_gate(g, e, 1)
    assert lec.dtype == torch.int64 and pos.dtype == torch.int64
    assert np.array_equal(lec.cpu().numpy(), ref_cnt)
    assert np.array_equal(pos.cpu().numpy(), ref_pos)
    assert gec is lec and all_ec is lec

    # the separate entry points, as fmoe/functions.py:19-42 strings them together
    cnt32 = torch.zeros(e, dtype=torch.int32, device=device)
    fmoe_native.expert_count(g, cnt32)
    fmoe_native.expert_count(g, cnt32)          # accumulates
    assert np.array_equal(cnt32.cpu().numpy(), 2 * ref_cnt)
    cum = torch.cumsum(torch.from_numpy(ref_cnt), 0).int().to(device)
    pos2 = torch.empty(int(ref_cnt.sum()), dtype=torch.int64, device=device)
    fmoe_native.assign_pos(cum, g, pos2)
    assert np.array_equal(pos2.cpu().numpy(), ref_pos)
    assert np.array_equal(cum.cpu().numpy(), (np.cumsum(ref_cnt) - ref_cnt).astype(np.int32))

    out = prepare_forward(g, e, 1)
    assert len(out) == 6 and all(not t.is_cuda for t in out[1:])
    assert np.array_equal(out[5].numpy(), ref_cnt)

    # the whole position buffer: routed slots first, -1 for the entries dropped slots leave unused
    cnt, pos_buf, s2r = fmoe_native.route(g, e)
    total = int(ref_cnt.sum())
    assert pos_buf.numel() == n * k and np.array_equal(pos_buf[:total].cpu().numpy(), ref_pos)
    assert bool((pos_buf[total:] == -1).all())


@pytest.mark.parametrize("n,k,e,cap", [(16384, 2, 16, 2458), (16384, 1, 64, 300), (8192, 8, 256, 100),
                                       (777, 2, 5, 0), (4096, 2, 8, 10 ** 6)])
def test_limit_and_prune_bit_exact(n, k, e, cap, device):
    rng = np.random.default_rng(cap % 1000 + n)
    gate = rng.integers(0, e, size=(n, k)).astype(np.int64)
    ref_lec, ref_gec, ref_pruned = orouting.limit_and_prune(gate, e, cap)
    g = torch.from_numpy(gate).to(device)
    new_lec, new_gec, pruned = limit_by_capacity(g, e, 1, cap)
    assert np.array_equal(new_gec.cpu().numpy(), ref_gec)
    assert np.array_equal(new_lec.cpu().numpy(), ref_lec)
    assert pruned.shape == g.shape and pruned.dtype == torch.int64
    assert np.array_equal(pruned.cpu().numpy(), ref_pruned)
    kept = np.bincount(ref_pruned[ref_pruned >= 0], minlength=e)
    assert np.all(kept <= cap)                       # tests/test_gates.py:51-57
    assert np.array_equal(g.cpu().numpy(), gate)     # input untouched, new tensor returned


def test_limit_by_capacity_several_workers(device):
    rng = np.random.default_rng(11)
    e, w = 37, 5
    ec = rng.integers(0, 50, size=w * e).astype(np.int64)
    cap = rng.integers(0, 120, size=e).astype(np.int32)
    cap_ref = cap.copy()
    ref = orouting.limit_by_capacity(ec, cap_ref, e, w)
    cap_dev = torch.from_numpy(cap).to(device)
    got = fmoe_native.limit_by_capacity(torch.from_numpy(ec).to(device), cap_dev, e, w)
    assert np.array_equal(got.cpu().numpy(), ref)
    assert np.array_equal(cap_dev.cpu().numpy(), cap_ref)


def test_prune_with_existing_drops_and_state(device):
    rng = np.random.default_rng(5)
    e = 12
    gate = rng.integers(-1, e, size=5000).astype(np.int64)
    ec = rng.integers(0, 300, size=e).astype(np.int32)
    ec_ref = ec.copy()
    ref = orouting.prune_gate_by_capacity(gate, ec_ref)
    ec_dev = torch.from_numpy(ec).to(device)
    got = fmoe_native.prune_gate_by_capacity(torch.from_numpy(gate).to(device), ec_dev, e, 1)
    assert np.array_equal(got.cpu().numpy(), ref)
    assert np.array_equal(ec_dev.cpu().numpy(), ec_ref)


def test_full_size_invariants(device):
    """Size-independent properties at the largest configuration (65 536 slots, 256 experts)."""
    torch.manual_seed(0)
    logits = torch.randn(8192, 256) + 0.5 * torch.randn(256)
    gate = torch.topk(logits, 8, dim=-1).indices.to(device)
    cnt, pos_buf, s2r = fmoe_native.route(gate, 256)
    total = int(cnt.sum())
    pos = pos_buf[:total]
    flat = gate.view(-1)
    assert total == flat.numel()
    assert torch.equal(torch.sort(pos).values, torch.arange(total, device=device))
    experts_along_pos = flat[pos]
    assert bool((experts_along_pos[1:] >= experts_along_pos[:-1]).all())
    assert torch.equal(s2r[pos], torch.arange(total, device=device))
    assert torch.equal(cnt, torch.bincount(flat, minlength=256))
    # idempotence of pruning: pruning the pruned gate with the same caps changes nothing
    cap = torch.full((256,), 200, dtype=torch.int32, device=device)
    once = fmoe_native.prune_gate_by_capacity(gate, cap.clone(), 256, 1)
    twice = fmoe_native.prune_gate_by_capacity(once, cap.clone(), 256, 1)
    assert torch.equal(once, twice)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,e,k", [
    (32768, 8, 2),      # the Mixtral-like share
    (8192, 256, 8),     # the fine-grained layer
    (16384, 64, 1),     # top-1
    (16384, 16, 2),
    (1000, 5, 4),       # experts not a power of two, token count not a multiple of a workgroup's share
    (77, 1003, 8),      # rows that do not start on 16-byte boundaries
    (700, 300, 4),
    (3, 2, 2),          # every expert chosen
    (0, 4, 2),
])
def test_gate_topk_route(dtype, n, e, k, device):
    """fmoe_gate_topk_route against torch.topk (tie-free logits, choices by descending logit), the
    scores in both modes, and its expert counts / pos / slot_to_row against the CPU oracle run on
    the SAME index tensor; its backward against autograd through torch.topk and softmax."""
    from fastermoe_amd import fmoe_native
    gen = torch.Generator().manual_seed(n + e + k)
    # distinct values per token, exactly representable in every dtype: consecutive bfloat16 bit patterns
    # (0.0078 .. 2.6, alternating sign), in a random order per token
    table = (torch.arange(e, dtype=torch.int16) + 0x3C00).view(torch.bfloat16).float()
    table = table * (1 - 2 * (torch.arange(e) % 2)).float()
    base = table[torch.argsort(torch.rand(n, e, generator=gen), dim=1)] if n else torch.zeros(0, e)
    logits = base.to(dtype).to(device)
    assert torch.equal(logits.float().cpu(), base)
    for mode in (0, 1):
        idx, score, cnt, pos_buf, s2r = fmoe_native.gate_topk_route(logits, k, mode)
        want_val, want_idx = torch.topk(logits.float(), k, dim=-1, largest=True, sorted=True)
        assert torch.equal(idx, want_idx)
        want_score = torch.softmax(want_val, dim=-1) if mode == 1 else want_val
        if mode == 0:
            assert torch.equal(score.float(), want_score)
        else:
            assert torch.allclose(score.float(), want_score, rtol={torch.float32: 1e-5}.get(dtype, 1e-2), atol=1e-6)
        ref_pos, ref_cnt = orouting.count_by_gate(idx.cpu().numpy(), e)
        assert np.array_equal(cnt.cpu().numpy(), ref_cnt)
        total = int(ref_cnt.sum())
        assert total == n * k
        assert np.array_equal(pos_buf[:total].cpu().numpy(), ref_pos)
        inv = np.full(n * k, -1, dtype=np.int64)
        inv[ref_pos] = np.arange(total)
        assert np.array_equal(s2r.cpu().numpy(), inv)
        if n == 0:
            continue
        # backward: d(sum(score * g)) / d(logits)
        g = torch.randn(n, k, generator=gen).to(dtype).to(device)
        got = fmoe_native.gate_topk_backward(g, score, idx, e, mode)
        leaf = logits.float().clone().requires_grad_(True)
        val, _ = torch.topk(leaf, k, dim=-1, sorted=True)
        sc = torch.softmax(val, dim=-1) if mode == 1 else val
        (sc * g.float()).sum().backward()
        assert torch.allclose(got.float(), leaf.grad, rtol={torch.float32: 1e-5}.get(dtype, 2e-2), atol=1e-2 if dtype != torch.float32 else 1e-6)


def test_gate_topk_ties_go_to_the_lower_expert(device):
    from fastermoe_amd import fmoe_native
    logits = torch.zeros(9, 6, device=device)
    logits[:, 4] = 1.0
    idx, score, cnt, _, _ = fmoe_native.gate_topk_route(logits, 4, 0)
    assert idx.cpu().tolist() == [[4, 0, 1, 2]] * 9
    assert cnt.cpu().tolist() == [9, 9, 9, 0, 9, 0]
    with pytest.raises(ValueError):
        fmoe_native.gate_topk_route(logits, 3, 0)        # not a power of two: torch.topk + route instead


def test_naive_gate_hands_its_routing_to_the_layer(device):
    """NaiveGate's index tensor carries the routing computed with the top-k; the layer's routing step
    uses it only for that very tensor, unmodified, and recomputes otherwise."""
    from fastermoe_amd import functions
    from fastermoe_amd.gates import NaiveGate
    torch.manual_seed(8)
    gate = NaiveGate(32, 8, 1, top_k=2).to(device)
    x = torch.randn(500, 32, device=device)
    idx, val = gate(x)
    assert hasattr(idx, "_fmoe_route")
    pos_a, cnt_a, cnt_cpu_a, s2r_a = functions._route(idx, 8, 1)
    fresh = idx.clone()
    assert not hasattr(fresh, "_fmoe_route")
    pos_b, cnt_b, _, s2r_b = functions._route(fresh, 8, 1)
    assert torch.equal(pos_a, pos_b) and torch.equal(cnt_a, cnt_b) and torch.equal(s2r_a, s2r_b)
    idx[0, 0] = -1                                       # an in-place edit invalidates what rides on the tensor
    pos_c, cnt_c, _, _ = functions._route(idx, 8, 1)
    assert int(cnt_c.sum()) == 999
    # scores are differentiable: the gate's weight gets a gradient through the selected logits
    idx2, val2 = gate(x)
    val2.sum().backward()
    assert gate.gate.weight.grad is not None and torch.isfinite(gate.gate.weight.grad).all()
    logits = gate.gate(x)
    # (the gate's linear layer ran inside the top-k kernel: same logits up to the order of the fp32 sums)
    assert torch.allclose(val2, torch.gather(logits, 1, idx2), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("e,k", [(8, 8), (64, 4), (65, 8), (250, 8), (256, 2), (513, 8), (8192, 8)])
def test_gate_topk_orders_equal_and_special_logits(dtype, e, k, device):
    """Many equal logits, both zeros, infinities, NaN (as -inf) and the smallest subnormals: by descending logit, of equal ones the
    lower expert, as sorting the pairs gives on the CPU; the scores are the logits."""
    gen = torch.Generator().manual_seed(e + k)
    tiny = 2.0 ** {torch.float32: -149, torch.bfloat16: -133, torch.float16: -24}[dtype]
    pool = torch.tensor([0.0, -0.0, 1.5, -1.5, float("inf"), -float("inf"), float("nan"), tiny, -tiny, 3.0, -3.0], dtype=torch.float64)
    logits = pool[torch.randint(len(pool), (37, e), generator=gen)].to(dtype)
    logits[0] = -float("inf")
    logits[1] = torch.arange(e, dtype=torch.float64).neg().to(dtype)
    idx, score = fmoe_native.gate_topk_route(logits.to(device), k, 0)[:2]
    values = logits.double()
    values = torch.where(values.isnan(), torch.full_like(values, -float("inf")), values)
    want = torch.stack([torch.tensor(sorted(range(e), key=lambda i: (-row[i], i))[:k]) for row in values.tolist()])
    assert torch.equal(idx.cpu(), want)
    assert torch.equal(score.double().cpu(), values.gather(1, want))


def test_gate_topk_with_masked_out_logits(device):
    """Logits of -inf (experts masked out by a caller) and NaN: a token with fewer than top_k finite
    logits still names top_k distinct experts -- the finite ones first, then the lowest-numbered of
    the rest -- instead of -1, which the gates would feed to bincount / index_add."""
    from fastermoe_amd import fmoe_native
    ninf = float("-inf")
    logits = torch.tensor([[ninf, 2.0, ninf, ninf, 1.0, ninf],
                           [ninf, ninf, ninf, ninf, ninf, ninf],
                           [0.5, ninf, 3.0, float("nan"), ninf, -1.0]], device=device)
    idx, score, cnt, pos_buf, s2r = fmoe_native.gate_topk_route(logits, 4, 0)
    assert idx.cpu().tolist() == [[1, 4, 0, 2], [0, 1, 2, 3], [2, 0, 5, 1]]
    assert score[0, :2].cpu().tolist() == [2.0, 1.0] and torch.isinf(score[0, 2:]).all()
    ref_pos, ref_cnt = orouting.count_by_gate(idx.cpu().numpy(), 6)
    assert np.array_equal(cnt.cpu().numpy(), ref_cnt) and int(ref_cnt.sum()) == 12
    assert np.array_equal(pos_buf.cpu().numpy(), ref_pos)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,e,k,bias", [
    (32768, 4096, 8, 2, True),     # the Mixtral-like share's gate
    (4096, 512, 8, 2, True),       # the tiny fp32 layer's gate
    (16384, 2048, 64, 1, True),    # top-1 over 64 experts
    (16384, 1024, 16, 2, False),
    (1000, 72, 5, 4, True),        # experts not a multiple of 16, tokens not a multiple of a workgroup's share,
                                   # contraction not a multiple of a wave's step
    (33, 8, 2, 2, True),
    (16, 2048, 64, 8, False),      # one workgroup of 16 tokens, and one token into the second
    (17, 1032, 33, 4, True),
    (4097, 136, 17, 2, True),      # past the sizes that take 16 tokens to a workgroup
    (100, 264, 64, 8, True),
    (0, 64, 4, 2, True),
])
def test_gate_linear_topk_route(dtype, n, d, e, k, bias, device):
    """The gate's linear layer inside the top-k kernel (fmoe_gate_linear_topk_route) against
    nn.Linear + torch.topk: the logits, formed in float64 from the same operands and rounded to the
    element type, fix the selection for every token whose k+1 largest logits are further apart than
    the rounding of the two different summation orders can move them -- those tokens must match
    torch.topk exactly; the scores must be the (rounded) logits of whatever was selected; and the
    routing must be the oracle's on the same index tensor, bit for bit."""
    from fastermoe_amd import fmoe_native
    gen = torch.Generator().manual_seed(n + d + e)
    x = torch.randn(n, d, generator=gen).to(dtype)
    w = (torch.randn(e, d, generator=gen) * (3.0 / d ** 0.5)).to(dtype)
    b = torch.randn(e, generator=gen).to(dtype) if bias else None
    xd, wd, bd = x.to(device), w.to(device), (b.to(device) if bias else None)
    ref = x.double() @ w.double().t()
    if bias:
        ref = ref + b.double()
    for mode in (0, 1):
        idx, score, cnt, pos_buf, s2r = fmoe_native.gate_linear_topk_route(xd, wd, bd, k, mode)
        assert idx.shape == (n, k) and score.dtype == dtype
        ref_pos, ref_cnt = orouting.count_by_gate(idx.cpu().numpy(), e)
        assert np.array_equal(cnt.cpu().numpy(), ref_cnt) and int(ref_cnt.sum()) == n * k
        assert np.array_equal(pos_buf.cpu().numpy(), ref_pos)
        inv = np.full(n * k, -1, dtype=np.int64)
        inv[ref_pos] = np.arange(n * k)
        assert np.array_equal(s2r.cpu().numpy(), inv)
        if n == 0:
            continue
        got_idx = idx.cpu()
        assert (got_idx.sort(dim=1).values.diff(dim=1) > 0).all() if k > 1 else True   # distinct experts
        top_val, top_idx = torch.topk(ref, min(k + 1, e), dim=1, sorted=True)
        # (float32: the two fp32 summation orders differ by about sqrt(d) roundings of the partial sums)
        step = {torch.float32: 2.0 ** -22 * max(1.0, d ** 0.5), torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
        # choice j of a token is settled when its logit is clear of both neighbours in the sorted order
        gaps = top_val[:, :-1] - top_val[:, 1:]                                   # [n, k] (or [n, e-1])
        ok = gaps > 4 * step * top_val.abs().max(dim=1, keepdim=True).values.clamp(min=1.0)
        below = ok if ok.shape[1] == k else torch.cat([ok, torch.ones(n, 1, dtype=torch.bool)], dim=1)
        above = torch.cat([torch.ones(n, 1, dtype=torch.bool), ok[:, :k - 1]], dim=1)
        clear = above & below[:, :k]
        assert clear.float().mean() > 0.3
        assert torch.equal(got_idx[clear], top_idx[:, :k][clear])
        picked = torch.gather(ref, 1, got_idx)
        if mode == 0:
            want = picked
        else:
            want = torch.softmax(picked, dim=1)
        tol = {torch.float32: 1e-5, torch.bfloat16: 1.6e-2, torch.float16: 2e-3}[dtype]
        assert torch.allclose(score.double().cpu(), want, rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mode", [0, 1])
def test_gate_linear_topk_autograd(dtype, mode, device):
    """GateLinearTopK's backward against autograd through nn.Linear, a gather at the SAME indices
    and the softmax: gradients of the input, the weight and the bias."""
    from fastermoe_amd.functions import GateLinearTopK
    torch.manual_seed(12)
    n, d, e, k = 600, 96, 12, 4
    lin = torch.nn.Linear(d, e).to(dtype).to(device)
    x = torch.randn(n, d, device=device).to(dtype).requires_grad_(True)
    g = torch.randn(n, k, device=device).to(dtype)
    idx, score = GateLinearTopK.apply(x, lin.weight, lin.bias, k, mode)
    assert hasattr(idx, "_fmoe_route")
    (score * g).sum().backward()
    got = [x.grad.clone(), lin.weight.grad.clone(), lin.bias.grad.clone()]
    x64 = x.detach().double().requires_grad_(True)
    w64, b64 = lin.weight.detach().double().requires_grad_(True), lin.bias.detach().double().requires_grad_(True)
    val = torch.gather(x64 @ w64.t() + b64, 1, idx)
    sc = torch.softmax(val, dim=1) if mode == 1 else val
    (sc * g.double()).sum().backward()
    tol = TOL[dtype] if dtype != torch.float32 else 1e-5
    for a, r in zip(got, [x64.grad, w64.grad, b64.grad]):
        assert rel_err(a, r) <= tol


def test_naive_gate_uses_the_fused_linear_and_matches_the_unfused_one(device, monkeypatch):
    from fastermoe_amd.gates import NaiveGate
    torch.manual_seed(4)
    gate = NaiveGate(256, 16, 1, top_k=2).to(device)
    x = torch.randn(3000, 256, device=device)
    results = []
    for flag in ("1", "0"):
        monkeypatch.setenv("FMOE_GATE_LINEAR_FUSED", flag)
        gate.zero_grad()
        idx, val = gate(x)
        val.square().sum().backward()
        results.append((idx, val, gate.gate.weight.grad.clone(), gate.gate.bias.grad.clone()))
    assert torch.equal(results[0][0], results[1][0])            # random fp32 logits: no near-ties
    for a, b in zip(results[0][1:], results[1][1:]):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)
    # with all logits asked for, the gate runs the linear layer by itself
    idx3, val3, logits = gate(x, return_all_scores=True)
    assert logits.shape == (3000, 16) and torch.equal(idx3, results[1][0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,e,k", [
    (1, 8, 1, 1),            # one token, one chunk, one expert
    (31, 128, 4, 2),         # fewer tokens than a step takes, a whole column tile
    (64, 136, 16, 2),        # a column over the tile, all experts of a block
    (65, 120, 17, 4),        # a token over the step, an expert over the block
    (1000, 520, 33, 8),
    (4097, 256, 64, 1),      # several token ranges with a ragged last one
    (2500, 384, 100, 2),
    (3000, 1032, 256, 8),    # the most experts
])
def test_gate_grad_from_selected_scores(dtype, n, d, e, k, device):
    """fmoe_gate_weight_grad and fmoe_reduce_slots_gate against the dense products in float64.  Allowed per
    element: float32 sums (an ulp per term of the sum of absolute terms) and the rounding of the result."""
    torch.manual_seed(n + d + e)
    x, w = torch.randn(n, d).to(dtype), torch.randn(e, d).to(dtype)
    g = torch.randn(n, k).to(dtype)
    idx = torch.rand(n, e).topk(k, dim=1).indices
    n_rows = max(1, (n * k * 3) // 4)
    rows = torch.randn(n_rows, d).to(dtype)
    s2r = torch.full((n * k,), -1, dtype=torch.int64)
    s2r[torch.randperm(n * k)[:n_rows]] = torch.arange(n_rows)
    out_eps = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -11}[dtype]
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0   # half of float16's smallest step

    def near(got, want, mag, terms):
        err = (got.double().cpu() - want).abs()
        assert (err <= 2 * out_eps * want.abs() + terms * 2.0 ** -24 * mag + tiny).all(), float(err.max())

    xd, wd, gd, idxd = (t.to(device) for t in (x, w, g, idx))
    dense = torch.zeros(n, e, dtype=torch.float64).scatter_(1, idx, g.double())
    grad_w, grad_b = fmoe_native.gate_weight_grad(gd, idxd, xd, e, True)
    near(grad_w, dense.t() @ x.double(), dense.abs().t() @ x.double().abs(), n)
    near(grad_b, dense.sum(0), dense.abs().sum(0), n)
    again, none = fmoe_native.gate_weight_grad(gd, idxd, xd, e, False)
    assert none is None and torch.equal(again, grad_w)
    part, mag = dense @ w.double(), dense.abs() @ w.double().abs()
    near(fmoe_native.reduce_slots_gate(None, None, gd, idxd, wd), part, mag, k + 1)
    picked = torch.where((s2r >= 0).unsqueeze(1), rows.double()[s2r.clamp(min=0)], torch.zeros(1, dtype=torch.float64))
    near(fmoe_native.reduce_slots_gate(rows.to(device), s2r.to(device), gd, idxd, wd), part + picked.view(n, k, d).sum(1),
         mag + picked.abs().view(n, k, d).sum(1), 2 * k + 1)


def test_naive_gate_of_many_experts_matches_the_dense_backward(device, monkeypatch):
    """More experts than the fused linear takes: same choices, scores and gradients as with the linear layer apart."""
    from fastermoe_amd.gates import NaiveGate
    torch.manual_seed(5)
    gate = NaiveGate(256, 200, 1, top_k=8).to(device)
    x = torch.randn(1500, 256, device=device, requires_grad=True)
    results = []
    for flag in ("1", "0"):
        monkeypatch.setenv("FMOE_GATE_LINEAR_FUSED", flag)
        gate.zero_grad()
        x.grad = None
        idx, val = gate(x)
        val.square().sum().backward()
        results.append((idx, val, x.grad, gate.gate.weight.grad.clone(), gate.gate.bias.grad.clone()))
    assert torch.equal(results[0][0], results[1][0])
    for a, b in zip(results[0][1:], results[1][1:]):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("n_expert", [16, 128])   # the linear inside the routing call, and as a library product
def test_naive_gate_backward_can_be_differentiated_again(n_expert, device):
    """A penalty on the gradient of the input reaches the gate's weight, as through the linear layer apart.  Bound:
    float32 sums of 70 terms and a gradient rounded once."""
    from fastermoe_amd.gates import NaiveGate
    torch.manual_seed(n_expert)
    gate = NaiveGate(64, n_expert, 1, top_k=2).to(device)
    x = torch.randn(70, 64, device=device, requires_grad=True)
    idx, val = gate(x)
    grad_x, = torch.autograd.grad(val.sum(), x, create_graph=True)
    grad_x.square().sum().backward()
    w = gate.gate.weight.detach().double().cpu().requires_grad_(True)
    picked = torch.zeros(70, n_expert, dtype=torch.float64).scatter_(1, idx.cpu().view(70, 2), 1.0)
    (picked @ w).square().sum().backward()
    assert torch.allclose(gate.gate.weight.grad.double().cpu(), w.grad, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("own", [True, False])
def test_hooks_see_the_linear_layer_of_a_gate_of_many_experts(own, device):
    """A forward hook on the gate's linear layer, or one for all modules, is called with its logits, as before the gate of
    more than 64 experts took the layer's parameters straight."""
    from fastermoe_amd.gates import NaiveGate
    torch.manual_seed(8)
    gate = NaiveGate(64, 100, 1, top_k=2).to(device)
    x = torch.randn(30, 64, device=device)
    seen = []

    def hook(module, args, out):
        if module is gate.gate:
            seen.append(out.detach().clone())

    handle = (gate.gate.register_forward_hook(hook) if own
              else torch.nn.modules.module.register_module_forward_hook(hook))
    try:
        idx, val = gate(x)
    finally:
        handle.remove()
    assert len(seen) == 1 and torch.equal(seen[0].gather(1, idx.view(30, 2)), val)


@pytest.mark.parametrize("n,d,e,k", [(32768, 512, 4, 4), (16384, 1024, 16, 2), (4096, 512, 100, 2), (9000, 256, 256, 8), (40, 8, 1, 1)])
def test_float32_gate_bias_gradient_keeps_its_precision(n, d, e, k, device):
    """The gradient of the gate's bias is a sum over all tokens.  Added in double per range of tokens, rounded to float32
    once per range and once at the end, its error is a rounding or two: 2^-23 of the gradient in 2-norm.  (A
    float32 chain over the tokens of a range gives up to 1e-6.)"""
    g = torch.Generator(device=device).manual_seed(n + e)
    x = torch.randn(n, d, device=device, generator=g)
    grad = torch.randn(n, k, device=device, generator=g)
    idx = torch.rand(n, e, device=device, generator=g).topk(k, dim=1).indices
    _, grad_b = fmoe_native.gate_weight_grad(grad, idx, x, e, True)
    want = torch.zeros(n, e, dtype=torch.float64, device=device).scatter_(1, idx, grad.double()).sum(dim=0)
    assert (grad_b.double() - want).norm() <= 2.0 ** -23 * want.norm()


@pytest.mark.parametrize("dtype,n,d,k", [
    (torch.bfloat16, 8192, 2056, 1), (torch.float16, 8192, 2056, 2), (torch.bfloat16, 4096, 1032, 4),   # two pieces per wave
    (torch.float32, 8192, 1028, 1), (torch.float32, 8192, 1028, 2),                                     # four
    (torch.float32, 8192, 516, 4), (torch.bfloat16, 8192, 2056, 8),                                     # two; one
])
def test_gate_input_gradient_of_long_rows(dtype, n, d, k, device):
    """The gate's part of the input gradient where a wave takes several pieces of a row, at row lengths that leave the last wave
    of a row partly empty, alone and with the experts' rows; tokens that name fewer experts.  Allowed per element: float32
    sums and the rounding of the result."""
    e = 16
    g = torch.Generator(device=device).manual_seed(n + d + k)
    w, grad = torch.randn(e, d, device=device, generator=g).to(dtype), torch.randn(n, k, device=device, generator=g).to(dtype)
    idx = torch.rand(n, e, device=device, generator=g).topk(k, dim=1).indices
    idx[::7, k - 1] = -1
    rows = torch.randn(n * k, d, device=device, generator=g).to(dtype)
    s2r = torch.randperm(n * k, device=device, generator=g)
    s2r[::5] = -1
    out_eps = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -11}[dtype]
    dense = torch.zeros(n, e + 1, dtype=torch.float64, device=device).scatter_(1, idx + 1, grad.double())[:, 1:].contiguous()
    part, mag = dense @ w.double(), dense.abs() @ w.double().abs()
    picked = torch.where((s2r >= 0).unsqueeze(1), rows.double()[s2r.clamp(min=0)], 0.0).view(n, k, d)
    for got, want, m in ((fmoe_native.reduce_slots_gate(None, None, grad, idx, w), part, mag),
                         (fmoe_native.reduce_slots_gate(rows, s2r, grad, idx, w), part + picked.sum(1), mag + picked.abs().sum(1))):
        assert bool(((got.double() - want).abs() <= 2 * out_eps * want.abs() + (2 * k + 1) * 2.0 ** -24 * m + 2.0 ** -25).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,e,k", [(300, 40, 12), (130, 256, 32), (70, 17, 17)])
def test_gate_weight_gradient_of_many_choices(n, e, k, dtype, device):
    """More choices per token than the entries that the weight gradient's kernel holds in registers from step to step."""
    d = 136
    g = torch.Generator(device=device).manual_seed(k)
    x, grad = torch.randn(n, d, device=device, generator=g).to(dtype), torch.randn(n, k, device=device, generator=g).to(dtype)
    idx = torch.rand(n, e, device=device, generator=g).topk(k, dim=1).indices
    dense = torch.zeros(n, e, dtype=torch.float64, device=device).scatter_(1, idx, grad.double())
    grad_w, grad_b = fmoe_native.gate_weight_grad(grad, idx, x, e, True)
    eps = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -9
    for got, want, mag in ((grad_w, dense.t() @ x.double(), dense.abs().t() @ x.double().abs()), (grad_b, dense.sum(0), dense.abs().sum(0))):
        assert bool(((got.double() - want).abs() <= 2 * eps * want.abs() + n * 2.0 ** -24 * mag).all())


def test_bytes_booked_for_the_gates_part(device):
    """The profile counts the rows that a pass reads and writes: not the experts' rows where it is given none."""
    import ctypes
    from fastermoe_amd import _lib
    lib = _lib.load()
    n, e, d, k = 256, 8, 512, 2
    w, grad = torch.randn(e, d, device=device), torch.randn(n, k, device=device)
    idx = torch.rand(n, e, device=device).topk(k, dim=1).indices
    rows, s2r = torch.randn(n * k, d, device=device), torch.arange(n * k, device=device)
    classes = lib.fmoe_profile_classes()
    for args, want in (((None, None), (n + e) * d * 4), ((rows, s2r), (k + 1) * n * d * 4)):
        launches, ms, work = (ctypes.c_int64 * classes)(), (ctypes.c_double * classes)(), (ctypes.c_double * classes)()
        _lib.check(lib.fmoe_profile_enable(1))
        fmoe_native.reduce_slots_gate(*args, grad, idx, w)
        _lib.check(lib.fmoe_profile_collect(*(ctypes.cast(a, ctypes.c_void_p) for a in (launches, ms, work)), classes))
        _lib.check(lib.fmoe_profile_enable(0))
        assert launches[6] == 1 and work[6] == want


@pytest.mark.parametrize("n,e,cap", [(1, 1, 0), (1, 4, 1), (64, 8, 3), (1000, 300, 2), (4097, 65, 64), (8192, 16, 1 << 30), (8192, 16, 400),
                                     (8193, 64, 100), (40000, 1024, 40), (32768, 16, 2458), (5000, 8, 0)])
@pytest.mark.parametrize("routed", [False, True])
def test_limit_and_route_in_one_call(n, e, cap, routed, device):
    """Counts, kept slots, their routing and the segment table under a capacity against the oracle and the routing of the pruned
    indices, bit for bit; with the indices' routing at hand and without; entries that name no expert among them."""
    from fastermoe_amd.functions import _attach_route, _route_launch
    from fastermoe_amd.gates.utils import limit_by_capacity
    rng = np.random.default_rng(n + e + cap)
    p = np.arange(1, e + 1) ** -0.7
    gate = rng.choice(e, size=n, p=p / p.sum()).astype(np.int64)
    gate[rng.random(n) < 0.1] = -1
    want_counts, _, want_idx = orouting.limit_and_prune(gate, e, cap)
    if n > 100:
        outside = rng.choice(np.flatnonzero(gate == -1), 2, replace=False)
        gate[outside] = [e, 1 << 40]
    idx = torch.from_numpy(gate).to(device)
    if routed:
        _attach_route(idx, e, *fmoe_native.route_table(idx, e))
    counts, again, pruned = limit_by_capacity(idx, e, 1, cap)
    assert counts is again and counts.dtype == torch.int64
    assert np.array_equal(counts.cpu().numpy(), want_counts)
    assert np.array_equal(pruned.cpu().numpy(), want_idx)
    got = _route_launch(pruned, e, with_table=True)
    assert got[0] is counts   # (the routing on the indices, not another one)
    fresh = fmoe_native.route_table(pruned, e)
    for a, b in zip(got[:3], fresh[:3]):
        assert torch.equal(a, b)
    rows, ints = int(want_counts.sum()), lambda t: t.cpu().numpy()
    table, ref = ints(got[3]), ints(fresh[3])
    assert table[1] == rows
    head = 8 + 3 * (e + 1)
    assert np.array_equal(table[:head], ref[:head])
    for tiles, at in ((2, 4), (3, 5)):
        lo, hi = table[at], table[at] + 4 * table[tiles]
        assert np.array_equal(table[lo:hi], ref[lo:hi])
    assert np.array_equal(table[-4 * e:], ref[-4 * e:])
    counts.zero_()   # a caller's own use of the counts: the routing is made anew
    assert torch.equal(_route_launch(pruned, e)[0], fresh[0])
    _, _, bare = limit_by_capacity(idx.view(1, -1), e, 1, cap)
    bare.fill_(0)    # and so it is after a write to the indices
    assert int(_route_launch(bare, e)[0][0]) == n


def test_capacity_of_gates_without_tokens_or_with_many_experts(device):
    from fastermoe_amd.gates.utils import limit_by_capacity
    counts, _, pruned = limit_by_capacity(torch.empty(0, 2, dtype=torch.int64, device=device), 4, 1, 3)
    assert counts.tolist() == [0] * 4 and pruned.shape == (0, 2)
    idx = torch.arange(3000, device=device) % 1500
    counts, _, pruned = limit_by_capacity(idx, 1500, 1, 1)
    assert counts.eq(1).all() and pruned[1500:].eq(-1).all() and torch.equal(pruned[:1500], idx[:1500])
