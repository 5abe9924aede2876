"""Next-token cross-entropy without the full logits tensor (the reference's adambridge/losses.py API).

The output projection of a large-vocabulary model turns [batch, seq, hidden] activations into
[batch, seq, vocab] logits -- gigabytes in FP32 for a 150k vocabulary -- which training then
keeps for the backward pass.  ``causal_lm_loss`` projects a slice of positions at a time and,
with gradients enabled, recomputes each slice's logits in the backward pass instead of keeping
them, so at most one slice of logits exists at once.

On the GPU a slice's cross-entropy and its gradient each are one pass of the library's kernels over
the logits as the head wrote them (csrc/abh_loss.hip).  Elsewhere, and wherever the slice is being
traced or differentiated in another way than one backward pass (:func:`_kernels_apply`), it is the
composition of torch operations, which defines the values.
"""

from __future__ import annotations

from typing import Callable

import torch
import torch.autograd.forward_ad as forward_ad
import torch.nn.functional as F
from torch.utils._device import DeviceContext
from torch.utils.checkpoint import checkpoint

from . import _hip

__all__ = ["causal_lm_loss"]


_MAX_ROWS = 1 << 23   # adambridge_cross_entropy's


# The kernels give each row a workgroup, which is mostly idle for a short one: from some number of rows on, torch's
# softmax, several short rows a workgroup, is faster.  (Rows up to which the kernels are taken whatever
# the vocabulary, and the vocabulary from which they are taken whatever the rows.)  Measured on MI355X, us,
# kernels / torch operations.  A slice's loss alone, BF16: 2^14 rows of 2 to 2048 values 97-122 / 98-165;
# 2^15 x 256 124 / 105; 2^16 x 2 153 / 95, x 256 200 / 153, x 512 216 / 226; 2^20 x 8 1893 / 770, x 512 3501 /
# 3447; FP32: 2^15 x 512 144 / 124, x 1000 185 / 186, 2^17 x 512 496 / 450, x 1000 671 / 730.  A training pass of
# a bare Linear head, with its other savings, BF16: 2^16 x 2 593 / 616, x 128 609 / 753; 2^17 x 8 856 / 758, x 128
# 1058 / 891, x 256 1136 / 1218; 2^18 x 256 1979 / 2335; FP32: 2^16 x 2 544 / 726; 2^17 x 256 1200 / 1186, 2^18 x 512
# 2930 / 3215.
_SLICE_RULE = (1 << 14, {torch.bfloat16: 512, torch.float32: 1000})
_HEAD_RULE = (1 << 16, {torch.bfloat16: 256, torch.float32: 512})


def _long_enough(rule: tuple, rows: int, vocab: int, dtype: torch.dtype) -> bool:
    return rows <= rule[0] or vocab >= rule[1][dtype]


def _observed() -> bool:
    """Whether something needs the torch operations themselves: a trace or compilation, a function
    transform (vmap, functorch grad), forward-mode derivatives, a mode that observes operations (a
    default device does not: it is where factory calls that name no device put their tensors)."""
    return bool(torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._are_functorch_transforms_active()
                or forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack()
                or any(not isinstance(torch._C._get_function_stack_at(i), DeviceContext)
                       for i in range(torch._C._len_torch_function_stack())))


def _ordinary(values: torch.Tensor, target: torch.Tensor) -> bool:
    """Whether rows of ``values`` and their ``target`` are plain contiguous tensors of the kernels' types on
    one GPU."""
    return (type(target) is torch.Tensor and values.is_cuda and target.device == values.device
            and values.dtype in (torch.bfloat16, torch.float32) and target.dtype == torch.int64
            and values.dim() == 2 and target.dim() == 1 and target.numel() == values.shape[0]
            and values.is_contiguous() and target.is_contiguous() and not values.is_neg()
            and 0 < values.shape[0] <= _MAX_ROWS and values.shape[1] > 0)


def _kernels_apply(logits: torch.Tensor, target: torch.Tensor, observed: bool | None = None) -> bool:
    """Whether the library's cross-entropy takes this slice (``observed``: :func:`_observed`, if asked before)."""
    return (not (_observed() if observed is None else observed) and type(logits) is torch.Tensor and _ordinary(logits, target)
            and _long_enough(_SLICE_RULE, *logits.shape, logits.dtype)
            and logits.data_ptr() % 16 == 0)   # so that the gradient, a new tensor, shares its alignment


def _head_applies(head, h: torch.Tensor, targets: torch.Tensor, chunk: int = 1) -> bool:
    """Whether ``head(h)`` is exactly ``h @ head.weight.T`` on plain tensors, so that :class:`_HeadLoss` may
    take the products itself: a torch.nn.Linear without a bias, with nothing hooked, replaced or cast
    around its call."""
    if type(head) is not torch.nn.Linear or head.bias is not None or "forward" in head.__dict__ or _observed():
        return False
    hooks = torch.nn.modules.module
    if (head._forward_hooks or head._forward_pre_hooks or head._backward_hooks or head._backward_pre_hooks
            or hooks._global_forward_hooks or hooks._global_forward_pre_hooks or hooks._global_backward_hooks
            or hooks._global_backward_pre_hooks or torch.is_autocast_enabled("cuda")):
        return False
    w = head.weight
    return (type(h) in (torch.Tensor, torch.nn.Parameter) and type(w) in (torch.Tensor, torch.nn.Parameter)
            and _ordinary(h, targets) and w.device == h.device and w.dtype == h.dtype and w.dim() == 2
            and w.is_contiguous() and not w.is_neg() and w.shape[1] == h.shape[1] and w.shape[0] > 0
            and _long_enough(_HEAD_RULE, min(chunk, h.shape[0]), w.shape[0], w.dtype))


def _plain_backward(gout: torch.Tensor) -> bool:
    """Whether this backward pass may run the kernels: not one that is differentiated in turn (create_graph)
    or observed, nor one whose incoming gradient is a batch (is_grads_batched) or otherwise holds no memory."""
    return (not torch.is_grad_enabled() and not _observed() and type(gout) is torch.Tensor
            and torch._C._has_storage(gout) and not gout._is_zerotensor())


def _logits_gradient(logits: torch.Tensor, target: torch.Tensor, ignore_index: int, gout: torch.Tensor) -> torch.Tensor:
    """What ``cross_entropy_backward`` computes, in torch operations: differentiable, and for a ``gout`` that is
    a batch (vmap)."""
    vocab = logits.shape[1]
    p = logits.float().softmax(1)
    hot = torch.arange(vocab, device=target.device) == target[:, None]
    seed = torch.where((target < 0) | (target >= vocab), torch.nan, gout)   # no such class: no gradient
    seed = torch.where(target == ignore_index, 0.0, seed)[:, None]          # an ignored row: 0 times what it holds
    return ((p - hot.float()) * seed).to(logits.dtype)


class _SliceLoss(torch.autograd.Function):
    """Summed cross-entropy by the library's kernels.  What is kept for the backward pass is the logits
    themselves and two floats per row."""

    @staticmethod
    def forward(ctx, logits, target, ignore_index):
        loss, stats = _hip.load().cross_entropy(logits, target, ignore_index)
        ctx.save_for_backward(logits, target, stats)
        ctx.ignore_index = ignore_index
        return loss

    @staticmethod
    def backward(ctx, gout, *_):
        logits, target, stats = ctx.saved_tensors
        if not _plain_backward(gout):
            return _logits_gradient(logits, target, ctx.ignore_index, gout), None, None
        return _hip.load().cross_entropy_backward(logits, target, ctx.ignore_index, stats, gout), None, None


class _SliceLossInTransform(_SliceLoss):
    """The same in the form that may run while a function transform is active, on tensors that are no part of
    it: a checkpointed slice computed again in a backward pass under vmap.  (A call of this form costs
    the host 30 us more.)"""

    @staticmethod
    def forward(logits, target, ignore_index):
        return _hip.load().cross_entropy(logits, target, ignore_index)

    @staticmethod
    def setup_context(ctx, inputs, output):
        logits, target, ctx.ignore_index = inputs
        ctx.save_for_backward(logits, target, output[1])
        ctx.mark_non_differentiable(output[1])
        ctx.set_materialize_grads(False)

    @staticmethod
    def vmap(info, in_dims, logits, target, ignore_index):
        raise NotImplementedError("batched logits take the torch operations (_kernels_apply)")


def _matmul_into(out: torch.Tensor, a: torch.Tensor, b: torch.Tensor) -> None:
    """``out`` = ``a @ b``: by the library's split product (csrc/abh_gemm.hip) where the inner dimension is long
    and the result small -- there the BLAS library leaves most of the chip idle -- else by torch.  (Measured
    where the lines lie, us, own / library: 8192 x 512 over 151936 terms 1460 / 1354, 4096 x 512 731 / 883, 4096 x
    896 1316 / 1374, 1024 x 4096 1354 / 1809; over 32000, 4096 x 896 291 / 320; over 16384, 4096 x 896 159 / 130,
    2048 x 2048 163 / 141, 4096 x 512 99 / 112, 2048 x 896 88 / 103.)"""
    (m, k), n = a.shape, b.shape[1]
    if (a.dtype == b.dtype == out.dtype == torch.bfloat16 and 1 << 14 <= k <= 1 << 22
            and m <= 4096 and m * n <= (1 << 22 if k >= 1 << 15 else 1 << 21) and n % 4 == 0 and k % 8 == 0
            and a.data_ptr() % 16 == 0 and b.data_ptr() % 8 == 0 and out.data_ptr() % 8 == 0):
        _hip.load().matmul(a, b, out)
    else:
        torch.mm(a, b, out=out)


class _HeadLoss(torch.autograd.Function):
    """Summed cross-entropy of ``h @ weight.T``, ``chunk`` rows at a time.  The backward pass computes each
    slice's logits again, as the checkpointed slices do, but no gradient beside them (it takes the
    logits' place), and the weight's gradient is added up inside the products (rounded once per slice,
    where the slices' gradients were each rounded, then added and rounded).

    The weight may have been written meanwhile (an optimizer step between two losses' backward passes;
    the update kernels write it without a version count): as in the checkpointed slices, the
    gradient is then that at the weight as it is, so the rows' statistics are taken from the logits
    computed again, and the weight is held by reference, not as a saved tensor."""

    @staticmethod
    def forward(ctx, h, weight, targets, ignore_index, chunk):
        k = _hip.load()
        total = h.new_zeros((), dtype=torch.float32)
        for h_part, t_part in zip(torch.split(h, chunk), torch.split(targets, chunk)):
            total += k.cross_entropy(torch.mm(h_part, weight.t()), t_part, ignore_index)[0]
        ctx.save_for_backward(h, targets)
        ctx.weight, ctx.ignore_index, ctx.chunk = weight, ignore_index, chunk
        return total

    @staticmethod
    def backward(ctx, gout):
        (h, targets), weight = ctx.saved_tensors, ctx.weight
        wanted = ctx.needs_input_grad[:2]
        parts = zip(torch.split(h, ctx.chunk), torch.split(targets, ctx.chunk))
        with torch.autocast(h.device.type, enabled=False):   # as the forward ran (_head_applies)
            if not _plain_backward(gout):
                dh, dw = [], 0.0
                for h_part, t_part in parts:
                    grad = _logits_gradient(torch.mm(h_part, weight.t()), t_part, ctx.ignore_index, gout)
                    if wanted[0]:
                        dh.append(torch.mm(grad, weight))
                    if wanted[1]:
                        dw = dw + torch.mm(grad.t(), h_part)
                return torch.cat(dh) if wanted[0] else None, dw if wanted[1] else None, None, None, None
            k = _hip.load()
            dh = torch.empty_like(h) if wanted[0] else None
            dw = None
            for (h_part, t_part), dh_part in zip(parts, torch.split(h if dh is None else dh, ctx.chunk)):
                logits = torch.mm(h_part, weight.t())
                stats = k.cross_entropy(logits, t_part, ctx.ignore_index)[1]
                grad = k.cross_entropy_backward(logits, t_part, ctx.ignore_index, stats, gout, out=logits)
                if wanted[0]:
                    _matmul_into(dh_part, grad, weight)
                if wanted[1]:
                    dw = torch.mm(grad.t(), h_part) if dw is None else dw.addmm_(grad.t(), h_part)
                del logits, grad
        return dh, dw, None, None, None


def _torch_loss_sum(logits: torch.Tensor, target: torch.Tensor, ignore_index: int) -> torch.Tensor:
    """Summed cross-entropy, logits upcast to FP32."""
    return F.cross_entropy(logits.float(), target, ignore_index=ignore_index, reduction="sum")


def _slice_loss_sum(h: torch.Tensor, target: torch.Tensor, project: Callable[[torch.Tensor], torch.Tensor],
                    ignore_index: int, observed: bool | None = None) -> torch.Tensor:
    """Summed cross-entropy of one slice.  A checkpointed slice is computed again in the backward pass, where
    other modes may be active but the same tensors must be saved: its caller passes what it found
    ``observed``."""
    logits = project(h)
    if not _kernels_apply(logits, target, observed):
        return _torch_loss_sum(logits, target, ignore_index)
    if torch.is_grad_enabled() and logits.requires_grad:
        if torch._C._are_functorch_transforms_active():
            return _SliceLossInTransform.apply(logits, target, ignore_index)[0]
        return _SliceLoss.apply(logits, target, ignore_index)
    return _hip.load().cross_entropy(logits, target, ignore_index)[0]


def causal_lm_loss(hidden_states: torch.Tensor, lm_head: Callable[[torch.Tensor], torch.Tensor],
                   labels: torch.Tensor, *, chunk_tokens: int = 1024, ignore_index: int = -100) -> torch.Tensor:
    """Mean next-token cross-entropy of ``lm_head(hidden_states)`` against ``labels``, evaluated
    ``chunk_tokens`` positions at a time (reference adambridge/losses.py:27-70).

    Position ``t`` is scored against ``labels[:, t + 1]`` (the last position of each sequence has
    no target); the mean runs over positions whose target is not ``ignore_index`` -- the Hugging
    Face causal-LM loss.  ``hidden_states``: ``[batch, seq, hidden]``; ``lm_head``: a module or
    function mapping ``[n, hidden]`` to ``[n, vocab]``; ``labels``: ``[batch, seq]`` token ids.
    With a gradient to the hidden states, each slice runs under non-reentrant ``torch.utils.checkpoint``,
    or (a plain ``torch.nn.Linear`` head on the GPU) in one function of the same memory
    (:class:`_HeadLoss`); with one to the head alone, the slices' logits are kept.
    """
    if hidden_states.dim() != 3:
        raise ValueError(f"hidden_states must be [batch, seq, hidden], got shape {tuple(hidden_states.shape)}")
    if tuple(labels.shape) != tuple(hidden_states.shape[:2]):
        raise ValueError(f"labels must be [batch, seq] = {tuple(hidden_states.shape[:2])}, got {tuple(labels.shape)}")
    if isinstance(chunk_tokens, bool) or not isinstance(chunk_tokens, int) or chunk_tokens < 1:
        raise ValueError("chunk_tokens must be a positive int")
    b, s, d = hidden_states.shape
    h = hidden_states.reshape(b * s, d)
    # targets: each sequence shifted left by one, its last position ignored
    targets = torch.full((b, s), ignore_index, dtype=labels.dtype, device=labels.device)
    targets[:, :-1] = labels[:, 1:]
    targets = targets.reshape(-1).to(h.device)
    n_scored = (targets != ignore_index).sum()
    recompute = torch.is_grad_enabled() and h.requires_grad
    if recompute and _head_applies(lm_head, h, targets, chunk_tokens):
        return _HeadLoss.apply(h, lm_head.weight, targets, ignore_index, chunk_tokens) / n_scored.clamp(min=1)
    observed = _observed()
    total = h.new_zeros((), dtype=torch.float32)
    for h_part, t_part in zip(torch.split(h, chunk_tokens), torch.split(targets, chunk_tokens)):
        if recompute:
            total = total + checkpoint(_slice_loss_sum, h_part, t_part, lm_head, ignore_index, observed,
                                       use_reentrant=False)
        else:
            total = total + _slice_loss_sum(h_part, t_part, lm_head, ignore_index, observed)
    return total / n_scored.clamp(min=1)
