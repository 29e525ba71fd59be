r"""MoE feed-forward block of a transformer (fmoe/transformer.py)."""
import os

import torch
import torch.nn as nn

from . import _lib, fmoe_native
from .functions import MOEExpertMLP, MOERoutedMLP, layer_call, nothing_watches
from .gates import NaiveGate
from .layers import FMoE, FMoELinear


class _Expert(nn.Module):
    r"""All experts of a worker as two grouped linears around an activation
    (fmoe/transformer.py:10-30)."""

    def __init__(self, num_expert, d_model, d_hidden, activation, rank=0, bias=True):
        super().__init__()
        self.htoh4 = FMoELinear(num_expert, d_model, d_hidden, bias=bias, rank=rank)
        self.h4toh = FMoELinear(num_expert, d_hidden, d_model, bias=bias, rank=rank)
        self.activation = activation

    def forward(self, inp, fwd_expert_count):
        # GELU (exact), ReLU or no activation: one autograd node with the activation in the GEMM
        # epilogues (FMOE_EXPERT_EPILOGUE=0 keeps the three modules apart, as the reference runs them)
        code = self._epilogue_activation()
        # (float64 keeps torch's activation: the epilogue's GELU is evaluated in single precision)
        if (code is not None and inp.is_cuda and inp.dtype in (torch.float32, torch.bfloat16, torch.float16)
                and os.environ.get("FMOE_EXPERT_EPILOGUE", "1") != "0"):
            return MOEExpertMLP.apply(inp, fwd_expert_count, self.htoh4.weight, self.htoh4.bias,
                                      self.h4toh.weight, self.h4toh.bias, code)
        x = self.htoh4(inp, fwd_expert_count)
        x = self.activation(x)
        return self.h4toh(x, fwd_expert_count)

    def routed_forward(self, inp, pos_buf, slot_to_row, counts_dev, top_k, table=None):
        r"""The experts over token rows ``inp [N, d_model]`` routed by ``pos_buf`` / ``slot_to_row`` /
        ``counts_dev`` (the device tensors of the routing call, and ``table``, the segment table of the
        counts, where the call made one), without any of them being read on the host: returns the
        experts' output in expert-sorted order, one row per slot, or ``None`` when this shape or
        activation needs the module-by-module path."""
        if not self._device_tables_apply(inp):
            return None
        code = self._epilogue_activation()
        if table is None:
            table = fmoe_native.segment_table(counts_dev, pos_buf.numel())
        params = (self.htoh4.weight, self.htoh4.bias, self.h4toh.weight, self.h4toh.bias)
        save = torch.is_grad_enabled() and (inp.requires_grad or any(p is not None and p.requires_grad for p in params))
        return MOERoutedMLP.apply(inp, *params, pos_buf, slot_to_row, table, top_k, code, save)

    def routed_layer(self, inp, gate_w, gate_b, score, routing, top_k):
        r"""The layer's output from its input as one call: with the gate's linear layer ``gate_w``, ``gate_b`` inside it, or
        over the ``score`` and ``routing`` (``pos_buf``, ``slot_to_row`` and the segment table) of a gate outside.  ``None``
        where that call does not apply: a subclass, replaced linears, another activation, tensors or sizes that it does not
        take, or somebody who watches the operators."""
        first, second = self._modules.get("htoh4"), self._modules.get("h4toh")
        if type(self) is not _Expert or type(first) is not FMoELinear or type(second) is not FMoELinear:
            return None
        try:
            params = [linear._parameters[name] for linear in (first, second) for name in ("weight", "bias")]
        except KeyError:   # (parametrised, or a view that a sharding wrapper put there)
            return None
        code = self._epilogue_activation()
        if code is None or params[0] is None or params[2] is None or not nothing_watches(inp, *(t for t in (gate_w, gate_b, score, *params) if t is not None)):
            return None
        if gate_w is None:
            gate = _lib.GATE_ROUTED
        elif fmoe_native.gate_linear_supported(inp.shape[1], gate_w.shape[0], top_k, inp.dtype):
            gate = _lib.GATE_LINEAR
        else:
            gate = _lib.GATE_LOGITS
        return layer_call(inp, gate_w, gate_b, score, *params, routing, top_k, code, gate)

    def unchunked_is_faster(self, inp, n_slots):
        r"""Whether :meth:`routed_forward` beats the chunked pipeline: where both linears run on the persistent
        kernel and nobody asks for a number of chunks.  The pipeline hides the row permutes behind the
        products of its chunks, but needs the counts on the host and pays every chunk's last round of tiles."""
        if "FMOE_FUSE_GRAN" in os.environ or not self._device_tables_apply(inp):
            return False
        n_expert, d_hidden, d_model = self.htoh4.weight.shape
        code = self._epilogue_activation()
        return (fmoe_native.linear_dev_reads_rows(n_slots, n_expert, d_model, d_hidden, inp.dtype, code, code == _lib.ACT_GELU)
                and fmoe_native.linear_dev_reads_rows(n_slots, n_expert, d_hidden, d_model, inp.dtype))

    def _device_tables_apply(self, inp):
        r"""Whether the products over a device table take these tensors.  They want whole 16-byte chunks on
        16-byte boundaries, in the sizes and in where the tensors begin: parameters that are views into one flat
        buffer, or rows that begin inside another tensor, go the module's or the pipeline's way instead."""
        d_hidden, d_model = self.htoh4.weight.shape[1:]
        return (self._epilogue_activation() is not None and inp.is_cuda
                and inp.dtype in (torch.float32, torch.bfloat16, torch.float16)
                and self.htoh4.weight.dtype == inp.dtype and self.h4toh.weight.dtype == inp.dtype
                and os.environ.get("FMOE_EXPERT_EPILOGUE", "1") != "0"
                and os.environ.get("FMOE_DEVICE_TABLES", "1") != "0"
                and fmoe_native.linear_dev_supported(d_model, d_hidden, inp.dtype)
                and all(t is None or t.data_ptr() % 16 == 0 for t in
                        (inp, self.htoh4.weight, self.htoh4.bias, self.h4toh.weight, self.h4toh.bias)))

    def _epilogue_activation(self):
        from .fused_functions import _activation_code
        try:
            return _activation_code(self.activation)
        except NotImplementedError:
            return None


def _gen_policy(alpha):
    r"""Shadowing policy factory (fmoe/transformer.py:33-87).  Shadowing copies
    experts between workers; with one worker the policy selects nothing."""

    def _no_policy(all_experts_count, all_global_expert_count, num_expert, world_size, d_model, fused):
        return all_experts_count.new_zeros(world_size, num_expert, dtype=bool)

    return _no_policy


class FMoETransformerMLP(FMoE):
    r"""``Linear(d_model, d_hidden) -> activation -> Linear(d_hidden, d_model)`` per
    expert, any leading input shape (fmoe/transformer.py:89-139)."""

    def __init__(self, num_expert=32, d_model=1024, d_hidden=4096, world_size=1, mp_group=None,
                 moe_group=None, activation=torch.nn.GELU(), gate=NaiveGate, top_k=2,
                 expert_dp_comm="none", gate_hook=None, bias=True, mask=None, mask_dict=None):
        super().__init__(num_expert=num_expert, d_model=d_model, gate=gate, top_k=top_k,
                         world_size=world_size, mp_group=mp_group, moe_group=moe_group,
                         gate_hook=gate_hook, mask=mask, policy_fn=_gen_policy(d_hidden / d_model),
                         mask_dict=mask_dict)
        self.experts = _Expert(num_expert, d_model, d_hidden, activation, rank=self.mp_rank, bias=bias)
        self.mark_parallel_comm(expert_dp_comm)

    def forward(self, inp: torch.Tensor):
        if inp.dim() == 2 and inp.shape[1] == self.d_model:
            return super().forward(inp)
        original_shape = inp.shape
        inp = inp.reshape(-1, self.d_model)
        output = super().forward(inp)
        return output.reshape(original_shape)
