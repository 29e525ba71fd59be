r"""Autograd Functions and routing helpers of the MoE layer, with the interface of
the reference's ``fmoe.functions`` (fmoe/functions.py), on top of
:mod:`fastermoe_amd.fmoe_native`.

Single worker only: ``world_size > 1`` (token all-to-all, dynamic shadowing) is
outside this package and raises ``NotImplementedError``.
"""
import torch
from torch.autograd import Function
from torch.utils._device import DeviceContext

from . import _lib, fmoe_native


def _single_worker(world_size, what):
    if world_size != 1:
        raise NotImplementedError(
            f"{what}: world_size={world_size}; this package implements the single-GPU "
            "path only (no global exchange, no dynamic shadowing)")


def ensure_comm(t, comm):
    """fmoe/functions.py:14-17 binds an NCCL communicator; nothing to do for one worker."""
    return None


def _whole_chunks(t):
    """Whether ``t`` lies as the kernels over 16-byte chunks read it: contiguous, beginning on 16 bytes."""
    return t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0)


def _as_chunks(t):
    """``t``, or a copy of it that satisfies :func:`_whole_chunks`.  What a forward saved does, but saved-tensor hooks may
    hand back anything equal to it (a view into the buffer that an offloader packed it into)."""
    return t if _whole_chunks(t) else t.clone(memory_format=torch.contiguous_format)


def _attach_route(idx, n_expert, counts, pos_buf, slot_to_row, table=None):
    """Leaves the routing (and segment table) of a gate's indices on them for :func:`_route_launch`, with the versions of
    the tensor that they are of and of the counts, which capacity helpers hand out.  Tensors made under ``torch.inference_mode`` count no versions, so a later write to
    them would go unseen: those are routed anew."""
    if not idx.is_inference():
        idx._fmoe_route = ((idx._version, counts._version), n_expert, counts, pos_buf, slot_to_row)
        idx._fmoe_table = table


class GateTopK(Function):
    r"""``torch.topk`` of the gate logits (and, with ``score_mode`` 1, the softmax over the selected
    logits) of fmoe/gates/naive_gate.py:26-42 with the routing of ``count_by_gate`` computed in
    the same launches.  Returns ``(topk_idx [N,k], topk_score [N,k])``; the routing result rides
    on ``topk_idx`` (``_fmoe_route``) and is picked up by :func:`_route` when the layer is handed
    this very tensor, unmodified."""

    @staticmethod
    def forward(ctx, logits, top_k, score_mode):
        logits = logits.contiguous()
        idx, score, cnt, pos_buf, s2r, table = fmoe_native.gate_topk_route(logits, top_k, score_mode, with_table=True)
        ctx.save_for_backward(idx, score)
        ctx.moe_args = logits.shape[1], score_mode
        ctx.mark_non_differentiable(idx)
        _attach_route(idx, logits.shape[1], cnt, pos_buf, s2r, table)
        return idx, score

    @staticmethod
    def backward(ctx, _grad_idx, grad_score):
        idx, score = ctx.saved_tensors
        n_expert, score_mode = ctx.moe_args
        return fmoe_native.gate_topk_backward(grad_score.contiguous(), score, idx, n_expert, score_mode), None, None


class GateLinearTopK(Function):
    r"""``nn.Linear`` -> ``torch.topk`` (-> softmax) of fmoe/gates/naive_gate.py:26-42 and the routing of
    ``count_by_gate`` in one call that keeps the logits on chip.  Returns ``(topk_idx, topk_score)`` like
    :class:`GateTopK`; the routing rides on ``topk_idx``.  Gates of more experts than that call takes, or with 16-bit rows
    off the 16-byte grid, run the linear layer as a library product first.  Backward: straight from the gradient of the selected logits; a softmax over
    them, a shape these kernels do not take, or ``create_graph`` goes through the dense gradient of the logits and library products."""

    @staticmethod
    def forward(ctx, x, weight, bias, top_k, score_mode):
        x = x.contiguous()
        weight = weight.contiguous()
        if fmoe_native.gate_linear_supported(x.shape[1], weight.shape[0], top_k, x.dtype):
            idx, score, cnt, pos_buf, s2r, table = fmoe_native.gate_linear_topk_route(x, weight, bias, top_k, score_mode,
                                                                                      with_table=True)
        else:
            idx, score, cnt, pos_buf, s2r, table = fmoe_native.gate_topk_route(
                torch.nn.functional.linear(x, weight, bias), top_k, score_mode, with_table=True)
        ctx.save_for_backward(x, weight, idx, score)
        ctx.moe_args = score_mode, bias is not None
        ctx.mark_non_differentiable(idx)
        _attach_route(idx, weight.shape[0], cnt, pos_buf, s2r, table)
        return idx, score

    @staticmethod
    def backward(ctx, _grad_idx, grad_score):
        x, weight, idx, score = ctx.saved_tensors
        score_mode, has_bias = ctx.moe_args
        grad_score = grad_score.contiguous()
        # (a backward that is to be differentiated again needs the products as torch operators)
        if (score_mode == 0 and not torch.is_grad_enabled() and _whole_chunks(x) and _whole_chunks(weight)
                and fmoe_native.gate_grad_any_supported(x.shape[1], weight.shape[0], idx.shape[1], x.dtype)):
            grad_x = grad_w = grad_b = None
            if ctx.needs_input_grad[0]:
                grad_x = fmoe_native.reduce_slots_gate(None, None, grad_score, idx, weight, any_grid=True)
            if ctx.needs_input_grad[1] or (has_bias and ctx.needs_input_grad[2]):
                grad_w, grad_b = fmoe_native.gate_weight_grad(grad_score, idx, x, weight.shape[0], has_bias, any_grid=True)
            return grad_x, grad_w, grad_b, None, None
        g = fmoe_native.gate_topk_backward(grad_score, score, idx, weight.shape[0], score_mode)
        grad_x = g @ weight if ctx.needs_input_grad[0] else None
        grad_w = g.t() @ x if ctx.needs_input_grad[1] else None
        grad_b = g.float().sum(dim=0).to(g.dtype) if has_bias and ctx.needs_input_grad[2] else None
        return grad_x, grad_w, grad_b, None, None


def _no_hooks(module):
    """Whether calling ``module`` is its class's ``forward`` and nothing else: no hook of its own, and none for
    all modules (profilers and debuggers register those)."""
    every = torch.nn.modules.module
    return ("forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                     or module._backward_pre_hooks or every._global_forward_hooks or every._global_forward_pre_hooks
                     or every._global_backward_hooks or every._global_backward_pre_hooks))


def _plain_linear(linear):
    """Whether calling ``linear`` is ``F.linear`` on its parameters and nothing else."""
    return type(linear) is torch.nn.Linear and _no_hooks(linear)


def gate_linear_topk(x, linear, top_k, score_mode=0):
    r"""Top-k indices and scores of ``linear(x)`` for an ``nn.Linear`` gate: one fused call when the
    shape is taken (CUDA tensors, at most 64 experts, ``top_k`` 1, 2, 4 or 8, rows of whole 16-byte
    chunks; ``FMOE_GATE_LINEAR_FUSED=0`` switches it off); one node over a library product where the gate's gradients take the shape
    (up to 256 experts, 16-bit rows of any length); else the layer followed by :func:`gate_topk`."""
    import os
    w, b = linear.weight, linear.bias
    if (x.is_cuda and x.dim() == 2 and w.is_cuda and w.dtype == x.dtype and (b is None or b.dtype == x.dtype)
            and os.environ.get("FMOE_GATE_LINEAR_FUSED", "1") != "0"
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0):
        if fmoe_native.gate_linear_supported(x.shape[1], w.shape[0], top_k, x.dtype):
            return GateLinearTopK.apply(x, w, b, top_k, score_mode)
        # more experts, or rows off the 16-byte grid: the library makes the logits, their gradient still is never formed
        if (_plain_linear(linear) and score_mode == 0 and x.shape[0] > 0 and not torch.is_autocast_enabled()
                and fmoe_native.gate_topk_supported(w.shape[0], top_k, x.dtype)
                and fmoe_native.gate_grad_any_supported(x.shape[1], w.shape[0], top_k, x.dtype)):
            return GateLinearTopK.apply(x, w, b, top_k, score_mode)
    return gate_topk(linear(x), top_k, score_mode)


class NoisyTopK(Function):
    r"""The training-mode selection of the noisy top-k gate (fmoe/gates/noisy_gate.py:113-144) after
    its two linear products: ``(topk_idx [N,k], gates [N,k], load [E])`` from the clean logits, the raw
    noise widths and a draw of N(0,1) noise, with the routing of ``count_by_gate`` riding on ``topk_idx``.
    ``load`` is the smooth estimate of tokens per expert (float32); both ``gates`` and ``load`` are
    differentiable with respect to ``clean`` and ``raw``."""

    @staticmethod
    def forward(ctx, clean, raw, noise, top_k, eps):
        clean, raw, noise = clean.contiguous(), raw.contiguous(), noise.contiguous()
        idx, gates, load, thr_val, thr_idx, cnt, pos_buf, s2r = fmoe_native.noisy_gate_forward(clean, raw, noise, top_k, eps)
        ctx.save_for_backward(clean, raw, noise, idx, gates, thr_val, thr_idx)
        ctx.moe_args = top_k, eps
        ctx.mark_non_differentiable(idx)
        _attach_route(idx, clean.shape[1], cnt, pos_buf, s2r)
        return idx, gates, load

    @staticmethod
    def backward(ctx, _grad_idx, grad_gates, grad_load):
        clean, raw, noise, idx, gates, thr_val, thr_idx = ctx.saved_tensors
        top_k, eps = ctx.moe_args
        if grad_gates is None:
            grad_gates = torch.zeros_like(gates)
        if grad_load is None:
            grad_load = torch.zeros(clean.shape[1], dtype=torch.float32, device=clean.device)
        g_clean, g_raw = fmoe_native.noisy_gate_backward(clean, raw, noise, top_k, eps, idx, gates, thr_val, thr_idx,
                                                         grad_gates.contiguous(), grad_load.float().contiguous())
        return g_clean, g_raw, None, None, None


def gate_topk(logits, top_k, score_mode=0):
    r"""Top-k indices and scores of ``logits [N, E]``: the HIP gate kernel when it takes the shape
    (CUDA tensor, 16/32-bit floats, ``top_k`` 1, 2, 4 or 8), ``torch.topk``
    otherwise.  ``score_mode`` 0: the selected logits; 1: their softmax over the ``top_k``."""
    if logits.is_cuda and logits.dim() == 2 and fmoe_native.gate_topk_supported(logits.shape[1], top_k, logits.dtype):
        idx, score = GateTopK.apply(logits, top_k, score_mode)
        # autograd hands back a new Python object for the index tensor: carry the routing over
        return idx, score
    val, idx = torch.topk(logits, k=top_k, dim=-1, largest=True, sorted=False)
    return idx, (torch.softmax(val, dim=-1) if score_mode == 1 else val)


def _route_launch(gate, num_expert, with_table=False):
    """Enqueues the routing of ``gate`` (or picks up the one its :class:`GateTopK` call made) and
    returns the device tensors ``(counts [E], pos_buf [n_slots], slot_to_row [n_slots])``; nothing
    is read back.  ``pos_buf`` holds the routed slots first and -1 after them.  ``with_table`` appends
    the segment table of the counts that the grouped GEMMs read."""
    with torch.no_grad():
        cached = getattr(gate, "_fmoe_route", None)
        if cached is not None and cached[0] == (gate._version, cached[2]._version) and cached[1] == num_expert:
            if not with_table:
                return cached[2:]
            table = getattr(gate, "_fmoe_table", None)
            if table is None:
                table = fmoe_native.segment_table(cached[2], cached[3].numel())
            return cached[2:] + (table,)
        routed = fmoe_native.route_table(gate.contiguous(), num_expert, with_table)
        return routed if with_table else routed[:3]


def _route(gate, num_expert, world_size):
    """(pos, counts, slot_to_row): one fused routing call and ONE device-to-host
    read (the counts), instead of the histogram / cumsum / ``.item()`` /
    placement sequence of fmoe/functions.py:19-42.  An index tensor that comes
    straight from :class:`GateTopK` carries its routing with it."""
    _single_worker(world_size, "count_by_gate")
    counts, pos_buf, slot_to_row = _route_launch(gate, num_expert)
    with torch.no_grad():
        counts_cpu = counts.cpu()
        pos = pos_buf[: int(counts_cpu.sum())]
    return pos, counts, counts_cpu, slot_to_row


class _PendingCounts:
    """The expert counts on their way to the host: an asynchronous copy into pinned memory that
    starts right behind the routing kernels.  ``counts_cpu`` is the CPU tensor the counts will be
    in; it carries this object as ``_fmoe_pending``, and whoever reads its values calls
    :meth:`wait` first (``fmoe_native`` does, just before a launch that needs them), so that all
    host work up to that point runs while the GPU is still busy with whatever precedes the
    routing, instead of after it.  Only the fused pipeline of this package's own expert module is
    handed such a tensor: it goes to the bindings unread."""

    # (thread, device, n_expert) -> [pinned int64 buffer, the _PendingCounts whose copy is in it or None]
    _staging = {}

    def __init__(self, counts):
        import threading
        key = (threading.get_ident(), counts.device.index, counts.numel())
        slot = self._staging.get(key)
        if slot is None:
            slot = self._staging[key] = [torch.empty(counts.numel(), dtype=torch.int64, pin_memory=True), None]
        elif slot[1] is not None:
            slot[1].wait()   # an earlier read-back that nobody has waited for yet still owns the buffer
        self._buf = slot[0]
        self._slot = slot
        self._done = False
        self.counts_cpu = torch.empty(counts.numel(), dtype=torch.int64)
        self.counts_cpu._fmoe_pending = self
        # the copy and the event go to the current stream of the counts' device, whichever device is current
        with torch.cuda.device(counts.device), torch.no_grad():
            self._buf.copy_(counts, non_blocking=True)
            self._event = torch.cuda.Event()
            self._event.record(torch.cuda.current_stream(counts.device))
        slot[1] = self

    def wait(self):
        if not self._done:
            self._event.synchronize()
            self.counts_cpu.copy_(self._buf)
            self._done = True
            if self._slot[1] is self:
                self._slot[1] = None
        return self.counts_cpu


def count_by_gate(gate, num_expert, world_size, require_pos=True):
    """fmoe/functions.py:19-42.  Returns ``(pos, local_expert_count,
    all_expert_count, global_expert_count, all_global_expert_count)``; with one
    worker the four count tensors are the same int64 ``[num_expert]`` tensor."""
    _single_worker(world_size, "count_by_gate")
    with torch.no_grad():
        if not require_pos:
            cnt32 = torch.zeros(num_expert, device=gate.device, dtype=torch.int32)
            fmoe_native.expert_count(gate.contiguous(), cnt32)
            counts = cnt32.long()
            pos = None
        else:
            pos, counts, _, _ = _route(gate, num_expert, world_size)
    return pos, counts, counts, counts, counts


def _prepare_forward_ex(gate, num_expert, world_size):
    pos, counts, counts_cpu, slot_to_row = _route(gate, num_expert, world_size)
    return (pos, counts_cpu, counts_cpu, counts_cpu, counts_cpu, counts_cpu.clone()), slot_to_row


def prepare_forward(gate, num_expert, world_size):
    r"""fmoe/functions.py:45-69: ``(pos, local_expert_count, global_expert_count,
    all_expert_count, all_global_expert_count, fwd_expert_count)`` with ``pos`` on
    the device and the counts on the CPU."""
    return _prepare_forward_ex(gate, num_expert, world_size)[0]


def _local_scatter(inp, pos):
    """fmoe/functions.py:72-74 (index_select)."""
    return fmoe_native.gather_rows(inp.contiguous(), pos)


def _local_gather(inp, pos, out_batch_size, maybe_overlap=True):
    """fmoe/functions.py:77-84: zero-fill then index_add_ (``maybe_overlap``) or
    index_copy_."""
    inp = inp.contiguous()
    if maybe_overlap:
        return fmoe_native.index_add_rows(inp, pos, out_batch_size)
    inverse = fmoe_native.invert_index(pos, out_batch_size)
    return fmoe_native.gather_rows(inp, inverse)


class MOECache(Function):
    r"""fmoe/functions.py:122-194.  The reference decides here which experts to
    shadow on other workers and raises for one worker; with one worker there is
    nothing to shadow, so this is the identity: ``models = [[experts]]``,
    ``stored_models`` all False, counts unchanged."""

    @staticmethod
    def forward(ctx, inp, all_expert_count, all_global_expert_count, local_expert_count,
                global_expert_count, fwd_expert_count, policy_fn, experts, batch_size, d_model,
                topk, num_expert, world_size, fused):
        _single_worker(world_size, "MOECache")
        stored_models = torch.zeros(world_size * num_expert, dtype=torch.bool)
        models = [[experts]] if fused else [experts]
        ctx.mark_non_differentiable(stored_models, fwd_expert_count)
        return inp.view_as(inp), models, stored_models, fwd_expert_count, int(fwd_expert_count.sum().item())

    @staticmethod
    def backward(ctx, grad_inp, *unused):
        return (grad_inp,) + (None,) * 13


class MOEScatter(Function):
    r"""Token rows -> expert-sorted rows (fmoe/functions.py:196-248).  ``pos`` is
    the token index of every sorted row (``pos // top_k``).  The two trailing
    arguments are optional extras: given ``slot_to_row`` and ``top_k`` the
    backward sums each token's ``top_k`` rows directly instead of going through
    the general index-add."""

    @staticmethod
    def forward(ctx, inp, pos, local_expert_count, global_expert_count, stored_models,
                fwd_batch_size, world_size, slot_to_row=None, top_k=None):
        _single_worker(world_size, "MOEScatter")
        buf = _local_scatter(inp, pos)
        ctx.moe_args = inp.shape[0], top_k
        ctx.save_for_backward(pos, slot_to_row)
        return buf

    @staticmethod
    def backward(ctx, grad_buf):
        pos, slot_to_row = ctx.saved_tensors
        n_tokens, top_k = ctx.moe_args
        grad_buf = grad_buf.contiguous()
        if slot_to_row is not None:
            grad_in = fmoe_native.reduce_slots(grad_buf, slot_to_row, n_tokens, top_k)
        else:
            grad_in = _local_gather(grad_buf, pos, n_tokens)
        return grad_in, None, None, None, None, None, None, None, None


class MOELinear(Function):
    r"""Per-expert linear over expert-sorted rows (fmoe/functions.py:251-275)."""

    @staticmethod
    def forward(ctx, global_input_buf, fwd_expert_count, weight, bias=None):
        global_input_buf = global_input_buf.contiguous()
        out = fmoe_native.linear_forward(global_input_buf, fwd_expert_count, weight, bias)
        ctx.save_for_backward(global_input_buf, fwd_expert_count, weight, bias)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        input_buf, fwd_expert_count, weight, bias = ctx.saved_tensors
        grad_in, grad_w, grad_b = fmoe_native.linear_backward(
            grad_out.contiguous(), input_buf, fwd_expert_count, weight, bias)
        return grad_in, None, grad_w, grad_b


class MOEExpertMLP(Function):
    r"""``Linear -> activation -> Linear`` of fmoe/transformer.py:22-30 over expert-sorted rows as
    one autograd node, so that the activation runs in the first GEMM's epilogue and its
    derivative in the epilogue of the second linear's data gradient, instead of as elementwise
    kernels over ``[rows, d_hidden]`` of their own.  ``activation`` is an ``ACT_*`` code
    (exact GELU, ReLU or none).  Not in the reference; same results as the three modules."""

    @staticmethod
    def forward(ctx, inp, fwd_expert_count, w1, b1, w2, b2, activation):
        from . import _lib
        inp = inp.contiguous()
        keep_pre = activation == _lib.ACT_GELU  # ReLU's derivative can be read off the output
        mid, pre = fmoe_native.linear_act_forward(inp, fwd_expert_count, w1, b1, activation, keep_pre)
        out = fmoe_native.linear_forward(mid, fwd_expert_count, w2, b2)
        ctx.save_for_backward(inp, fwd_expert_count, w1, b1, w2, b2, pre, mid)
        ctx.activation = activation
        return out

    @staticmethod
    def backward(ctx, grad_out):
        inp, fwd_expert_count, w1, b1, w2, b2, pre, mid = ctx.saved_tensors
        grad_out = grad_out.contiguous()
        g_pre = fmoe_native.linear_dact_backward(grad_out, fwd_expert_count, w2, pre if pre is not None else mid,
                                                 ctx.activation)
        gw2, gb2 = fmoe_native.linear_weight_backward(grad_out, mid, fwd_expert_count, w2, b2)
        g_inp, gw1, gb1 = fmoe_native.linear_backward(g_pre, inp, fwd_expert_count, w1, b1)
        return g_inp, None, gw1, gb1, gw2, gb2, None


class MOERoutedMLP(Function):
    r"""``MOEScatter`` -> ``Linear -> activation -> Linear`` (fmoe/functions.py:196-248,
    fmoe/transformer.py:22-30) over the rows as the routing kernels left them, with nothing read
    back to the host: all GEMMs take the experts' row segments from ``table``, the device-side segment
    table of the routing's counts.  Small first GEMMs read token row ``pos_buf[r] // top_k`` for
    sorted row ``r`` in their loader (no scattered copy in the forward); large ones run on a kernel that wants
    sorted rows.  The copy made for them is not kept for the first linear's weight gradient, which makes its own: the
    tokens, which the gate keeps anyway, are saved, not ``top_k`` times as many rows.  Returns the
    experts' output in expert-sorted order, one row per slot (``[n_slots, d_model]``; the rows past the
    routed ones are not written), for :class:`MOEGatherCombine` / :class:`MOEGather`.  With ``save`` false (nothing
    will be differentiated) the pre-activations are not written.
    Not in the reference; same results as ``MOEScatter`` + the three modules."""

    @staticmethod
    def forward(ctx, inp, w1, b1, w2, b2, pos_buf, slot_to_row, table, top_k, activation, save):
        from . import _lib
        inp = inp.contiguous()
        n_slots = pos_buf.numel()
        keep_pre = save and activation == _lib.ACT_GELU  # ReLU's derivative can be read off the output
        n_expert, d_hidden, d_model = w1.shape
        in_loader = (inp.numel() * inp.element_size() < (1 << 31)
                     and not fmoe_native.linear_dev_reads_rows(n_slots, n_expert, d_model, d_hidden, inp.dtype, activation, keep_pre))
        src = inp if in_loader else fmoe_native.gather_rows(inp, pos_buf, index_div=top_k)
        mid, pre = fmoe_native.linear_forward_dev(src, w1, b1, table, n_slots, activation, keep_pre,
                                                  row_index=pos_buf if in_loader else None, index_div=top_k)
        del src   # (its memory serves the output, which is as large)
        out, _ = fmoe_native.linear_forward_dev(mid, w2, b2, table, n_slots)
        if save:
            ctx.save_for_backward(inp, w1, b1, w2, b2, pos_buf, slot_to_row, table, pre, mid)
        ctx.moe_args = top_k, activation
        return out

    @staticmethod
    def backward(ctx, grad_out):
        inp, w1, b1, w2, b2, pos_buf, slot_to_row, table, pre, mid = map(_as_chunks, ctx.saved_tensors)
        top_k, activation = ctx.moe_args
        n_slots = pos_buf.numel()
        grad_out = grad_out.contiguous()
        g_pre = fmoe_native.linear_dgrad_dev(grad_out, w2, table, n_slots, pre if pre is not None else mid, activation)
        gw2, gb2 = fmoe_native.linear_wgrad_dev(grad_out, mid, w2, table, n_slots, b2 is not None)
        g_inp = None
        if ctx.needs_input_grad[0]:
            g_rows = fmoe_native.linear_dgrad_dev(g_pre, w1, table, n_slots)
            g_inp = fmoe_native.reduce_slots(g_rows, slot_to_row, inp.shape[0], top_k)
        rows = fmoe_native.gather_rows(inp, pos_buf, index_div=top_k)
        gw1, gb1 = fmoe_native.linear_wgrad_dev(g_pre, rows, w1, table, n_slots, b1 is not None)
        return g_inp, gw1, gb1, gw2, gb2, None, None, None, None, None, None


class MOELayer(Function):
    r"""The layer between its input and its output as one autograd node: gate (``routing`` ``None``: the linear layer
    ``gate_w``, ``gate_b`` and its top-k), :class:`MOERoutedMLP` and :class:`MOEGatherCombine`, each direction one call into
    the library.  With a gate outside, ``score`` and ``routing = (pos_buf, slot_to_row, table)`` are its results.
    Not in the reference; the same results as the nodes one by one, except that the gate's part of the input gradient is added
    before the sum is rounded."""

    @staticmethod
    def forward(ctx, inp, gate_w, gate_b, score, w1, b1, w2, b2, routing, top_k, activation, gate, sizes):
        inp = inp.contiguous()
        if routing is None:
            place = fmoe_native.LayerRouting.block(inp.shape[0] * top_k, sizes[2], inp.element_size(), inp.device)
        else:
            place = fmoe_native.LayerRouting(score, *routing)
        out, pre, mid, rows = fmoe_native.layer_forward(inp, gate_w, gate_b, _gate_logits(gate, inp, gate_w, gate_b), w1, b1, w2, b2,
                                                        top_k, activation, 1, gate, sizes, place)
        ctx.save_for_backward(inp, gate_w, w1, w2, pre, mid, rows, place.kept, *place.tensors)
        ctx.moe_args = top_k, activation, gate, sizes, [b is not None for b in (gate_b, b1, b2)]
        return out

    @staticmethod
    def backward(ctx, grad_out):
        inp, gate_w, w1, w2, pre, mid, rows, kept, *tensors = map(_as_chunks, ctx.saved_tensors)
        top_k, activation, gate, sizes, (gate_bias, bias1, bias2) = ctx.moe_args
        need = ctx.needs_input_grad
        place = fmoe_native.LayerRouting(*tensors, kept=kept)
        # (a backward that is to be differentiated again needs the gate's products as torch operators, and so do gates that the
        # kernels do not take)
        apart = kept is not None and (torch.is_grad_enabled() or not fmoe_native.gate_grad_any_supported(
            inp.shape[1], gate_w.shape[0], top_k, inp.dtype))
        new = lambda wanted, *shape: torch.empty(shape, dtype=inp.dtype, device=inp.device) if wanted else None
        (n, d), (e, h) = inp.shape, w1.shape[:2]
        grad_x = new(need[0], n, d)
        grad_score = new(kept is None or apart, n, top_k)
        gate_wanted = kept is not None and not apart and (need[1] or need[2])
        grad_gate_w, grad_gate_b = new(gate_wanted, e, d), new(gate_wanted and gate_bias, e)
        first, second = need[4] or need[5], need[6] or need[7]
        grad_w1, grad_b1 = new(first, e, h, d), new(first and bias1, e, h)
        grad_w2, grad_b2 = new(second, e, d, h), new(second and bias2, e, d)
        from ._lib import GATE_ROUTED
        fmoe_native.layer_backward(grad_out.contiguous(), inp, gate_w, w1, w2, top_k, activation, GATE_ROUTED if apart else gate, sizes, place,
                                   pre, mid, rows, grad_x, grad_score, grad_gate_w, grad_gate_b, grad_w1, grad_b1, grad_w2, grad_b2)
        if apart:
            idx, score = place.gate_results(n, top_k, sizes[2], inp.dtype)
            g = fmoe_native.gate_topk_backward(grad_score, score, idx, e, 0)
            grad_x = grad_x + g @ gate_w if need[0] else None
            grad_gate_w = g.t() @ inp if need[1] else None
            grad_gate_b = g.float().sum(dim=0).to(g.dtype) if gate_bias and need[2] else None
        return (grad_x, grad_gate_w, grad_gate_b, grad_score if kept is None else None, grad_w1, grad_b1, grad_w2, grad_b2,
                None, None, None, None, None)


def _gate_logits(gate, inp, gate_w, gate_b):
    """The logits of a gate whose linear layer stays a library product."""
    from ._lib import GATE_LOGITS
    return torch.nn.functional.linear(inp, gate_w, gate_b) if gate == GATE_LOGITS else None


def layer_call(inp, gate_w, gate_b, score, w1, b1, w2, b2, routing, top_k, activation, gate):
    r"""The layer's output through :class:`MOELayer`, or, where nothing will be differentiated, through the same call without
    a node; ``None`` where the call does not take these tensors (see :func:`fmoe_native.layer_sizes`)."""
    keep = torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (inp, gate_w, gate_b, score, w1, b1, w2, b2))
    if not keep and _lib.load_layer_call() is not None:
        return fmoe_native.layer_infer(inp, gate_w, gate_b, score, routing, w1, b1, w2, b2, top_k, activation, gate)
    n, d = inp.shape
    e, h = w1.shape[0], w1.shape[1]
    params = [t for t in (gate_w, gate_b, score, w1, b1, w2, b2) if t is not None]
    dtype, device = inp.dtype, inp.device
    for t in params:
        if t.dtype != dtype or t.device != device or not t.is_contiguous() or t.data_ptr() % 16 != 0:
            return None
    if (inp.data_ptr() % 16 != 0 or w1.shape != (e, h, d) or w2.shape != (e, d, h) or (b1 is not None and b1.shape != (e, h))
            or (b2 is not None and b2.shape != (e, d)) or (gate_w is not None and gate_w.shape != (e, d))
            or (gate_b is not None and gate_b.shape != (e,))):
        return None
    sizes = fmoe_native.layer_sizes(n, d, h, e, top_k, dtype, activation, int(keep), gate)
    if sizes is None:
        return None
    if not keep:
        inp = inp.contiguous()
        place = fmoe_native.LayerRouting() if routing is None else fmoe_native.LayerRouting(score, *routing)
        return fmoe_native.layer_forward(inp, gate_w, gate_b, _gate_logits(gate, inp, gate_w, gate_b), w1, b1, w2, b2, top_k, activation, 0,
                                         gate, sizes, place)[0]
    return MOELayer.apply(inp, gate_w, gate_b, score, w1, b1, w2, b2, routing, top_k, activation, gate, sizes)


def saving_is_watched():
    r"""Whether saved-tensor hooks are in force where something may be saved: an offloader's, or an activation checkpoint's, which
    compares what a forward and its second run save.  The second run may go without the hooks and modes of the first, so what is
    saved must not depend on them then."""
    return torch.is_grad_enabled() and torch._C._autograd._top_saved_tensors_default_hooks(True) is not None


def _modes_watch():
    """Whether a mode is in force that would have to see the operators: not one that only names the device of new tensors
    (``with torch.device(...)``, ``torch.set_default_device``)."""
    if torch._C._len_torch_dispatch_stack() != 0:
        return True
    return (torch._C._len_torch_function_stack() != 0
            and any(type(mode) is not DeviceContext for mode in torch.overrides._get_current_function_mode_stack()))


def nothing_watches(*tensors):
    r"""Whether a call on these tensors is seen by autograd's plain reverse mode at most: no transform (vmap, forward
    mode), trace, compiler, mode or tensor subclass that would have to see the operators of the layer one by one.  Modes count only
    where :func:`saving_is_watched` is false."""
    return (all(type(t) is torch.Tensor or type(t) is torch.nn.Parameter for t in tensors)
            and torch._C._functorch.peek_interpreter_stack() is None and torch.autograd.forward_ad._current_level < 0
            and torch._C._get_tracing_state() is None and not torch.compiler.is_compiling()
            and (not _modes_watch() or saving_is_watched()))


class MOEGather(Function):
    r"""Expert-sorted rows -> slot order, zero rows for dropped slots
    (fmoe/functions.py:278-330).  ``slot_to_row`` (optional extra) is the inverse
    of ``pos``; without it the inverse is rebuilt from ``pos``."""

    @staticmethod
    def forward(ctx, global_output_buf, pos, local_expert_count, global_expert_count,
                stored_models, local_batch_size, world_size, slot_to_row=None):
        _single_worker(world_size, "MOEGather")
        buf = global_output_buf.contiguous()
        if slot_to_row is None:
            slot_to_row = fmoe_native.invert_index(pos, local_batch_size)
        out = fmoe_native.gather_rows(buf, slot_to_row, local_batch_size)
        ctx.save_for_backward(pos)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        (pos,) = ctx.saved_tensors
        return _local_scatter(grad_out, pos), None, None, None, None, None, None, None


class MOECombine(Function):
    r"""``torch.bmm(gate_score[N,1,k], x[N,k,d])`` of fmoe/layers.py:321-322 as one
    streaming kernel (fp32 accumulation, one rounding) with its backward."""

    @staticmethod
    def forward(ctx, x, gate_score, n_tokens, top_k):
        x = x.contiguous()
        gate_score = gate_score.contiguous()
        ctx.save_for_backward(x, gate_score)
        ctx.moe_args = n_tokens, top_k, gate_score.shape
        return fmoe_native.combine_forward(x, gate_score, n_tokens, top_k)

    @staticmethod
    def backward(ctx, grad_out):
        x, gate_score = ctx.saved_tensors
        n_tokens, top_k, score_shape = ctx.moe_args
        grad_x, grad_score = fmoe_native.combine_backward(grad_out.contiguous(), x, gate_score, n_tokens, top_k)
        return grad_x, grad_score.view(score_shape), None, None


class MOEGatherCombine(Function):
    r"""``MOEGather`` (fmoe/functions.py:285-312) and the ``bmm`` with the gate scores
    (fmoe/layers.py:321-322) as one pass over the experts' output in expert-sorted
    order: ``out[t] = sum_j score[t,j] * rows[slot_to_row[t*k+j]]``; dropped slots
    (``slot_to_row < 0``) contribute zero, as the zero rows of ``_local_gather`` do."""

    @staticmethod
    def forward(ctx, rows, slot_to_row, gate_score, n_tokens, top_k):
        rows = rows.contiguous()
        gate_score = gate_score.contiguous()
        ctx.save_for_backward(rows, slot_to_row, gate_score)
        ctx.moe_args = n_tokens, top_k, gate_score.shape
        return fmoe_native.gather_combine_forward(rows, slot_to_row, gate_score, n_tokens, top_k)

    @staticmethod
    def backward(ctx, grad_out):
        rows, slot_to_row, gate_score = ctx.saved_tensors
        n_tokens, top_k, score_shape = ctx.moe_args
        grad_rows, grad_score = fmoe_native.gather_combine_backward(grad_out.contiguous(), rows, slot_to_row,
                                                                    gate_score, n_tokens, top_k)
        return grad_rows, None, grad_score.view(score_shape), None, None


def mask_index(mask):
    r"""For FMoE's ``mask`` (fmoe/layers.py:288-293): ``(keep_idx, token_to_row)`` -- the indices of
    the tokens whose mask is 0 (what ``inp[mask == 0]`` selects, here in descending token order)
    and, per token, its row among the kept ones (-1 for masked tokens).  One routing call with a
    single "expert" and one device-to-host read (the number of kept tokens), no boolean indexing."""
    with torch.no_grad():
        key = (mask.reshape(-1) != 0).to(torch.int64).neg_()        # 0: keep, -1: masked
        counts, pos_buf, token_to_row = fmoe_native.route(key, 1)
        keep_idx = pos_buf[: int(counts.cpu()[0])]
    return keep_idx, token_to_row


class MaskSelect(Function):
    r"""``rows[keep_idx]``: the rows of the kept tokens (``inp[mask == 0, :]``, fmoe/layers.py:292);
    the backward puts the gradient rows back and leaves zero rows for masked tokens."""

    @staticmethod
    def forward(ctx, rows, keep_idx, token_to_row):
        ctx.save_for_backward(token_to_row)
        return fmoe_native.gather_rows(rows.contiguous(), keep_idx)

    @staticmethod
    def backward(ctx, grad_rows):
        (token_to_row,) = ctx.saved_tensors
        return fmoe_native.gather_rows(grad_rows.contiguous(), token_to_row), None, None


class MaskRestore(Function):
    r"""Back to the full token order (fmoe/layers.py:305-317, with the combine of :322 already
    applied to the kept tokens): ``out[t] = kept[token_to_row[t]]`` for kept tokens and
    ``scale[t] * fill[fill_row[t]]`` for a masked token whose mask value has a ``mask_dict`` entry
    (``scale`` = the sum of the token's gate scores, since every one of its ``top_k`` slots holds
    the same ``mask_dict`` value), zero rows otherwise.  ``fill`` may be ``None``."""

    @staticmethod
    def forward(ctx, kept, keep_idx, token_to_row, scale, fill, fill_row):
        ctx.save_for_backward(keep_idx, token_to_row, scale, fill, fill_row)
        return fmoe_native.mask_restore(kept.contiguous(), token_to_row, scale, fill, fill_row, token_to_row.numel())

    @staticmethod
    def backward(ctx, grad_out):
        keep_idx, token_to_row, scale, fill, fill_row = ctx.saved_tensors
        grad_out = grad_out.contiguous()
        grad_kept = fmoe_native.gather_rows(grad_out, keep_idx)
        grad_scale = grad_fill = None
        if fill is not None and scale is not None and ctx.needs_input_grad[3]:
            grad_scale = fmoe_native.mask_scale_grad(grad_out, token_to_row, fill, fill_row)
        if fill is not None and ctx.needs_input_grad[4]:
            # a mask_dict value that is trained: rare, plain torch
            masked = (token_to_row < 0) & (fill_row >= 0)
            w = scale.float() if scale is not None else torch.ones_like(fill_row, dtype=torch.float32)
            contrib = (grad_out.float() * (w * masked).unsqueeze(1))
            grad_fill = torch.zeros(fill.shape, dtype=torch.float32, device=fill.device).index_add_(
                0, fill_row.clamp(min=0), contrib).to(fill.dtype)
        return grad_kept, None, None, grad_scale, grad_fill, None


class AllGather(Function):
    r"""fmoe/functions.py:333-349 (model-parallel group); one worker only."""

    @staticmethod
    def forward(ctx, inp, rank, world_size, group):
        _single_worker(world_size, "AllGather")
        return inp.view_as(inp)

    @staticmethod
    def backward(ctx, grad_out):
        return grad_out, None, None, None


class Slice(Function):
    r"""fmoe/functions.py:352-375 (model-parallel group); one worker only."""

    @staticmethod
    def forward(ctx, inp, rank, world_size, group):
        _single_worker(world_size, "Slice")
        return inp.view_as(inp)

    @staticmethod
    def backward(ctx, grad_out):
        return grad_out, None, None, None
