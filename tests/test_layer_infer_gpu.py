"""The layer's call for inference, from tensors to kernels in native code: what it takes, what it leaves to the steps, and where it fails."""
import pytest
import torch

from fastermoe_amd import _lib, fmoe_native, functions

pytestmark = pytest.mark.gpu


def tensors(device, n=5, d=64, h=128, e=4, dtype=torch.bfloat16):
    g = torch.Generator(device=device).manual_seed(3)
    new = lambda *s: torch.randn(*s, generator=g, device=device).to(dtype)
    return dict(inp=new(n, d), gate_w=new(e, d), gate_b=new(e), score=None, routing=None, w1=new(e, h, d), b1=new(e, h), w2=new(e, d, h), b2=new(e, d),
                top_k=2, activation=_lib.ACT_GELU, gate=_lib.GATE_LINEAR)


def test_it_takes_what_the_layer_gives_it(device):
    t = tensors(device)
    out = fmoe_native.layer_infer(**t)
    assert out.shape == t["inp"].shape and out.dtype == t["inp"].dtype and out.device == t["inp"].device and not out.requires_grad
    wide = torch.randn(5, 128, device=device).to(torch.bfloat16)
    wide[:, :64] = t["inp"]
    assert torch.equal(fmoe_native.layer_infer(**dict(t, inp=wide[:, :64])), out)   # rows that lie apart are copied
    logits = dict(t, gate=_lib.GATE_LOGITS)
    assert fmoe_native.layer_infer(**logits).shape == out.shape
    with torch.inference_mode():
        assert fmoe_native.layer_infer(**t).is_inference()


@pytest.mark.parametrize("name,change", [
    ("w1", lambda t: t.float()), ("b2", lambda t: t.cpu()), ("w2", lambda t: t.transpose(1, 2)), ("gate_w", lambda t: t[:, ::2]),
    ("b1", lambda t: t[:, :-8].contiguous()), ("gate_b", lambda t: torch.cat([t, t])[1:5]), ("inp", lambda t: t[0]),
    ("inp", lambda t: torch.cat([t.flatten(), t.flatten()])[1:1 + t.numel()].view_as(t)), ("w1", lambda t: t[:3]), ("top_k", lambda k: 9)])
def test_it_leaves_the_rest_to_the_steps(name, change, device):
    t = tensors(device)
    assert fmoe_native.layer_infer(**dict(t, **{name: change(t[name])})) is None


def test_a_failing_call_raises(device):
    with pytest.raises(_lib.FmoeHipError):
        fmoe_native.layer_infer(**dict(tensors(device), gate=_lib.GATE_ROUTED))   # no routing is given
    with pytest.raises(TypeError):
        fmoe_native.layer_infer(**dict(tensors(device), gate_w=1))


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 52), (torch.float32, 64)])
@pytest.mark.parametrize("outside", [False, True])
def test_without_the_extension_module_the_result_is_the_same(dtype, d, outside, device, monkeypatch):
    """The layer's call from Python: bit for bit, with the gate inside (off the 16-byte grid: its logits a library product) and outside."""
    gate = _lib.GATE_LINEAR if d % 8 == 0 else _lib.GATE_LOGITS
    t = tensors(device, d=d, dtype=dtype, h=128 if d % 8 == 0 else 100)
    if outside:
        idx, score = torch.randn(5, 4, device=device).topk(2).indices, torch.randn(5, 2, device=device).to(dtype)
        cnt, pos, slot_to_row = fmoe_native.route(idx, 4)
        t.update(gate_w=None, gate_b=None, score=score, routing=(pos, slot_to_row.view(-1), fmoe_native.segment_table(cnt, 10)))
        gate = _lib.GATE_ROUTED
    args = [t[k] for k in ("inp", "gate_w", "gate_b", "score", "w1", "b1", "w2", "b2", "routing", "top_k", "activation")] + [gate]
    with torch.no_grad():
        native = functions.layer_call(*args)
        monkeypatch.setattr(_lib, "_layer_call", None)
        assert native is not None and torch.equal(functions.layer_call(*args), native)
