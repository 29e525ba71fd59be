"""The layer as one call (``MOELayer`` / ``fmoe_layer_forward`` / ``fmoe_layer_backward``) against the same layer step by
step: the kernels are the same, so everything is equal bit by bit but the input's gradient, whose gate part is added before
the one rounding instead of after two."""
import contextlib
import copy

import pytest
import torch
import torch.utils.checkpoint

import fastermoe_amd as fmoe
from fastermoe_amd import _lib, fmoe_native, functions
from fastermoe_amd.gates import NaiveGate
from fastermoe_amd.gates.utils import limit_by_capacity

EPS = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}   # a whole rounding step


class Watching(torch.overrides.TorchFunctionMode):
    """Sees every operator and changes nothing: the layer then runs its steps one by one."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class DroppingGate(NaiveGate):
    def forward(self, inp):
        idx, score = super().forward(inp)
        return limit_by_capacity(idx, self.num_expert, 1, max(1, idx.numel() // (2 * self.num_expert)))[2], score


def build(device, dtype, d, h, e, k, act=None, bias=True, gate=NaiveGate, fuse=False):
    torch.manual_seed(d + h + e)
    with device:
        moe = fmoe.FMoETransformerMLP(num_expert=e, d_model=d, d_hidden=h, top_k=k, gate=gate, bias=bias,
                                      activation=act or torch.nn.GELU())
    moe = moe.to(dtype)
    moe.enable_fuse = fuse
    return moe


def step(moe, x, grad, watched):
    moe.zero_grad(set_to_none=True)
    x = x.detach().requires_grad_(x.requires_grad)
    if watched:
        with Watching():
            out = moe(x)
    else:
        out = moe(x)
    out.backward(grad)
    return out, x.grad, {n: p.grad for n, p in moe.named_parameters()}


def compare(moe, x, grad, calls, monkeypatch, rounded=()):
    """``rounded``: gradients that the steps round once more or add in another order."""
    seen = []
    real = functions.MOELayer.apply
    monkeypatch.setattr(functions.MOELayer, "apply", lambda *a: (seen.append(1), real(*a))[1])
    out, gx, grads = step(moe, x, grad, False)
    assert len(seen) == calls
    ref_out, ref_gx, ref_grads = step(moe, x, grad, True)
    assert len(seen) == calls
    assert torch.equal(out, ref_out)
    assert set(grads) == set(ref_grads)
    for name, g in grads.items():
        assert (g is None) == (ref_grads[name] is None), name
        if g is not None and name not in rounded:
            assert torch.equal(g, ref_grads[name]), name
        elif g is not None:
            err = (g.double() - ref_grads[name].double()).abs().max() / ref_grads[name].double().abs().max()
            assert err <= 2 * EPS[x.dtype], name
    assert (gx is None) == (ref_gx is None)
    if gx is not None:
        # two roundings of the parts and one of their sum against one: each at most half a step of the part or the sum, and
        # the parts exceed the sum only where they cancel, by no more than the largest part
        err = (gx.double() - ref_gx.double()).abs().max() / ref_gx.double().abs().max()
        assert err <= 2 * EPS[x.dtype]


SHAPES = [(1, 64, 128, 4, 1), (3, 64, 96, 32, 2), (257, 256, 512, 8, 2), (130, 128, 64, 65, 8), (300, 64, 64, 256, 4),
          (2048, 512, 1024, 8, 2), (4096, 1024, 2048, 16, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,d,h,e,k", SHAPES)
def test_one_call_equals_the_steps(dtype, n, d, h, e, k, device, monkeypatch):
    act = [torch.nn.GELU(), torch.nn.ReLU(), torch.nn.Identity()][(n + e) % 3]
    moe = build(device, dtype, d, h, e, k, act, bias=n != 257)
    x = torch.randn(n, d, device=device).to(dtype).requires_grad_(True)
    compare(moe, x, torch.randn(n, d, device=device).to(dtype), 1, monkeypatch)


ODD = [(1, 20, 30, 4, 1), (3, 7, 9, 3, 2), (257, 100, 130, 6, 2), (500, 64, 66, 8, 2), (500, 66, 64, 8, 2), (130, 321, 127, 70, 8),
       (2000, 500, 1302, 12, 2), (64, 1000, 2001, 300, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,h,e,k", ODD)
def test_feature_sizes_off_the_grid(dtype, n, d, h, e, k, device, monkeypatch):
    """16-bit types with rows that are no whole 16-byte chunks: the same call over a device table, against the steps over host
    counts; slots that a gate drops; inference."""
    act = [torch.nn.GELU(), torch.nn.ReLU(), torch.nn.Identity()][(n + e) % 3]
    x = torch.randn(n, d, device=device).to(dtype).requires_grad_(True)
    grad = torch.randn(n, d, device=device).to(dtype)
    moe = build(device, dtype, d, h, e, k, act, bias=n != 257)
    # (the linear layer's own backward rounds its bias gradient's sum in parts; with rows on the grid the gate has kernels)
    compare(moe, x, grad, 1, monkeypatch, rounded=("gate.gate.bias",))
    compare(build(device, dtype, d, h, e, k, act, gate=DroppingGate), x, grad, 1, monkeypatch, rounded=("gate.gate.bias",))
    with torch.no_grad():
        got = moe(x)
        with Watching():
            assert torch.equal(got, moe(x))


@pytest.mark.gpu
@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("n,d,h,e,k", [(513, 128, 256, 8, 2), (8192, 512, 2048, 16, 4), (203, 1544, 64, 12, 9), (65, 1032, 1304, 32, 17),
                                       (2048, 1024, 4096, 16, 2)])
def test_gate_outside_the_call(n, d, h, e, k, fuse, device, monkeypatch):
    """A gate that drops slots (none of expert rows may be read for them), and a hook on a plain one.  All memory that a pass allocates begins as
    NaN: the rows past the routed ones are written by nothing.  (The last size has 1024 tiles of 256 x 256 of weight gradients, on the persistent kernel.)"""
    real = torch.empty
    blank = lambda *a, **kw: real(*a, **kw).view(torch.uint8).fill_(255).view(kw["dtype"])
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: blank(*a, **kw) if kw.get("dtype") in (torch.uint8, torch.bfloat16)
                        and torch.device(kw.get("device", "cpu")).type == "cuda" else real(*a, **kw))
    x = torch.randn(n, d, device=device).to(torch.bfloat16).requires_grad_(True)
    grad = torch.randn(n, d, device=device).to(torch.bfloat16)
    moe = build(device, torch.bfloat16, d, h, e, k, gate=DroppingGate, fuse=fuse)
    one_call = not fuse or moe.experts.unchunked_is_faster(x, n * k)
    compare(moe, x, grad, int(one_call), monkeypatch)
    hooked = build(device, torch.bfloat16, d, h, e, k, fuse=fuse)
    got = []
    hooked.gate_hook = lambda idx, score, _: got.append((idx, score))
    compare(hooked, x, grad, int(one_call), monkeypatch)
    assert len(got) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_the_input_gradient_rounded_once_is_nearer_to_float64(dtype, device):
    """The sum of the experts' and the gate's part is rounded once, the steps round both parts and their sum."""
    n, d, h, e, k = 1500, 256, 512, 8, 2
    moe = build(device, dtype, d, h, e, k, torch.nn.ReLU())
    x = torch.randn(n, d, device=device).to(dtype).requires_grad_(True)
    grad = torch.randn(n, d, device=device).to(dtype)
    idx = moe.gate(x.detach())[0]
    exact = copy.deepcopy(moe).double()
    leaf = x.detach().double().requires_grad_(True)
    score, one, two = exact.gate.gate(leaf).gather(1, idx), exact.experts.htoh4, exact.experts.h4toh
    out = torch.zeros_like(leaf)
    for i in range(e):
        t, j = (idx == i).nonzero(as_tuple=True)
        y = torch.relu(leaf[t] @ one.weight[i].t() + one.bias[i]) @ two.weight[i].t() + two.bias[i]
        out = out.index_add(0, t, y * score[t, j][:, None])
    want, = torch.autograd.grad(out, leaf, grad.double())
    once, thrice = ((step(moe, x, grad, watched)[1].double() - want).norm() for watched in (False, True))
    assert once <= thrice


@pytest.mark.gpu
def test_partial_gradients_and_orders(device, monkeypatch):
    """Frozen experts, a frozen gate, an input without gradient, rows that are a transposed view, a 3-D input, gradients that
    begin off 16 bytes, two backwards of one forward."""
    n, d, h, e, k = 200, 128, 256, 8, 2
    dtype = torch.bfloat16
    moe = build(device, dtype, d, h, e, k)
    x = torch.randn(n, d, device=device).to(dtype)
    grad = torch.randn(n * d + 1, device=device).to(dtype)[1:].view(n, d)
    compare(moe, x, grad, 1, monkeypatch)
    for frozen in ("experts", "gate", "experts.htoh4", "experts.h4toh"):
        part = copy.deepcopy(moe)
        part.get_submodule(frozen).requires_grad_(False)
        compare(part, x.clone().requires_grad_(True), grad, 1, monkeypatch)
    turned = torch.randn(d, n, device=device).to(dtype).t().requires_grad_(True)
    compare(moe, turned, grad, 1, monkeypatch)
    three = torch.randn(4, 50, d, device=device).to(dtype)
    with torch.no_grad():
        assert torch.equal(moe(three), moe(three.reshape(200, d)).view(4, 50, d))
    leaf = x.clone().requires_grad_(True)
    out = moe(leaf)
    first, = torch.autograd.grad(out, leaf, grad, retain_graph=True)
    second, = torch.autograd.grad(out, leaf, grad)
    assert torch.equal(first, second)


@pytest.mark.gpu
def test_create_graph_reaches_the_gate(device):
    """Under ``create_graph`` the gate's part of the input gradient depends on the gate's weight, as with the steps apart."""
    n, d, h, e, k = 64, 64, 128, 8, 2
    moe = build(device, torch.float32, d, h, e, k)
    x = torch.randn(n, d, device=device)

    def second(watched):
        leaf = x.clone().requires_grad_(True)
        with (Watching() if watched else torch.enable_grad()):
            out = moe(leaf)
        gx, = torch.autograd.grad(out.square().sum(), leaf, create_graph=True)
        return gx, torch.autograd.grad(gx.square().sum(), moe.gate.gate.weight)[0]

    for got, want in zip(second(False), second(True)):
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5 * float(want.detach().abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("e", [8, 100])
def test_inference_takes_no_node_and_transforms_keep_theirs(e, device):
    n, d, h, k = 37, 64, 128, 2
    moe = build(device, torch.bfloat16, d, h, e, k)
    x = torch.randn(n, d, device=device).to(torch.bfloat16)
    with torch.no_grad():
        want = moe(x)
        with Watching():
            assert torch.equal(want, moe(x))
        with pytest.raises(Exception):   # (as before: no forward-mode formula, rather than a result without its tangent)
            with torch.autograd.forward_ad.dual_level(), torch.enable_grad():
                moe(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
    moe.requires_grad_(False)
    out = moe(x)
    assert not out.requires_grad and torch.equal(out, want)


class WatchingDispatch(torch.utils._python_dispatch.TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@contextlib.contextmanager
def module_hook():
    handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda module, args: None)
    try:
        yield
    finally:
        handle.remove()


@pytest.mark.gpu
@pytest.mark.parametrize("inside", ["forward", "backward"])
@pytest.mark.parametrize("watcher", ["device", "function mode", "dispatch mode", "module hook"])
def test_a_checkpointed_layer_saves_the_same_in_both_runs(watcher, inside, device):
    """The second run of a checkpoint does not see the modes and hooks that were in force around the first, or sees others."""
    make = {"device": lambda: torch.device("cuda"), "function mode": Watching, "dispatch mode": WatchingDispatch, "module hook": module_hook}[watcher]
    n, d, h, e, k = 96, 64, 128, 8, 2
    moe = build(device, torch.bfloat16, d, h, e, k)
    x = torch.randn(n, d, device=device).to(torch.bfloat16).requires_grad_(True)
    grad = torch.randn(n, d, device=device).to(torch.bfloat16)
    _, want, wants = step(moe, x, grad, False)
    moe.zero_grad(set_to_none=True)
    with (make() if inside == "forward" else contextlib.nullcontext()):
        out = torch.utils.checkpoint.checkpoint(moe, x, use_reentrant=False)
    with (make() if inside == "backward" else contextlib.nullcontext()):
        out.backward(grad)
    for name, p in moe.named_parameters():
        assert torch.equal(p.grad, wants[name]), name
    assert (x.grad.double() - want.double()).abs().max() <= 2 * EPS[torch.bfloat16] * want.double().abs().max()   # (as in compare)


@pytest.mark.gpu
def test_a_default_device_keeps_the_one_call(device, monkeypatch):
    moe = build(device, torch.bfloat16, 64, 128, 8, 2)
    x = torch.randn(5, 64, device=device).to(torch.bfloat16).requires_grad_(True)
    seen = []
    real = functions.MOELayer.apply
    monkeypatch.setattr(functions.MOELayer, "apply", lambda *a: (seen.append(len(a[8] or ())), real(*a))[1])
    with torch.device(device):
        moe(x)
    assert seen == [0]   # (the gate inside)


def test_what_watches():
    t = torch.zeros(1)
    hooks = lambda: torch.autograd.graph.saved_tensors_hooks(lambda v: v, lambda v: v)
    assert functions.nothing_watches(t) and not functions.saving_is_watched()
    with torch.device("cpu"):
        assert functions.nothing_watches(t)
        with Watching():
            assert not functions.nothing_watches(t)
            with hooks():
                assert functions.nothing_watches(t) and functions.saving_is_watched()
    with WatchingDispatch():
        assert not functions.nothing_watches(t)
    with hooks(), torch.no_grad():
        assert not functions.saving_is_watched()


def test_sizes_say_what_is_taken(monkeypatch):
    """Host only: sizes grow with what is kept apart, shapes that a step does not take and switches that keep the steps apart
    are refused."""
    f = fmoe_native.layer_sizes
    bf16 = torch.bfloat16
    fwd, bwd, table = f(100, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_LINEAR)
    assert bwd == 0 and table == _lib.load().fmoe_segment_table_bytes(200, 8) and fwd >= 200 * (64 + 128) * 2
    assert f(100, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 1, _lib.GATE_LINEAR)[1] >= 200 * (64 + 128) * 2
    assert f(100, 64, 128, 8, 2, torch.float64, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is None
    assert f(100, 60, 130, 8, 2, bf16, _lib.ACT_GELU, 1, _lib.GATE_ROUTED) is not None   # rows of 120 bytes: 16-bit types
    assert f(100, 60, 130, 8, 2, bf16, _lib.ACT_GELU, 1, _lib.GATE_LINEAR) is None       # (not by the kernel of the gate's linear layer)
    assert f(100, 60, 130, 8, 2, bf16, _lib.ACT_GELU, 1, _lib.GATE_LOGITS) is not None
    assert f(100, 62, 128, 8, 2, torch.float32, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is None
    assert f(0, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is None
    assert f(100, 64, 128, 100, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_LINEAR) is None   # more experts than the gate kernel holds
    assert f(100, 64, 128, 100, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_LOGITS) is not None
    assert f(100, 64, 128, 100, 3, bf16, _lib.ACT_GELU, 0, _lib.GATE_LOGITS) is None
    assert f(100, 64, 128, 100, 3, bf16, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is not None
    for name in ("FMOE_FOLD_COMBINE", "FMOE_EXPERT_EPILOGUE", "FMOE_DEVICE_TABLES"):
        monkeypatch.setenv(name, "0")
        assert f(100, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is None
        monkeypatch.delenv(name)
    monkeypatch.setenv("FMOE_GATE_LINEAR_FUSED", "0")
    assert f(100, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_LINEAR) is None
    assert f(100, 64, 128, 8, 2, bf16, _lib.ACT_GELU, 0, _lib.GATE_ROUTED) is not None
