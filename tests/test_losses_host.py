"""causal_lm_loss's choice between the library's kernels and torch operations, and its backward passes'
surroundings, on the CPU: the kernels are stood in for by torch operations that refuse any operand the
real ones could not take."""

import pytest
import torch
import torch.nn.functional as F

import adambridge_amd as ab
from adambridge_amd import _hip, losses

IGNORE = -100


class Kernels:
    """HipKernels' loss calls in torch operations on host tensors; ``calls`` names each one made."""

    def __init__(self):
        self.calls = []

    def cross_entropy(self, logits, target, ignore_index):
        self.calls.append("cross_entropy")
        assert type(logits) is torch.Tensor and logits.dtype in (torch.float32, torch.bfloat16)
        logits.data_ptr()
        x = logits.detach().float()
        m = x.amax(1)
        s = (x - m[:, None]).exp().sum(1)
        at = target.clamp(0, x.shape[1] - 1)[:, None]
        terms = torch.where(target == ignore_index, 0.0, s.log() - (x.gather(1, at)[:, 0] - m))
        return terms.sum(), torch.stack((m, 1.0 / s), 1)

    def cross_entropy_backward(self, logits, target, ignore_index, stats, gout, out=None):
        self.calls.append("cross_entropy_backward")
        assert gout.dtype == torch.float32 and gout.numel() == 1
        logits.data_ptr(), gout.data_ptr()
        g = torch.where(target == ignore_index, 0.0, gout)[:, None]
        p = (logits.detach().float() - stats[:, :1]).exp() * stats[:, 1:] * g
        p.scatter_add_(1, target.clamp(0, p.shape[1] - 1)[:, None], -g)
        out = torch.empty_like(logits) if out is None else out
        assert out.dtype == logits.dtype and out.shape == logits.shape
        return out.copy_(p)

    def matmul(self, a, b, out):
        self.calls.append("matmul")
        assert a.dtype == b.dtype == out.dtype == torch.bfloat16
        out.copy_(a.float() @ b.float())


@pytest.fixture
def kernels(monkeypatch):
    """The stand-ins, taken for host tensors as the real ones are for tensors on a GPU."""
    def ordinary(values, target):
        return (type(target) is torch.Tensor and values.dtype in (torch.bfloat16, torch.float32)
                and target.dtype == torch.int64 and values.dim() == 2 and target.dim() == 1
                and target.numel() == values.shape[0] and values.is_contiguous() and target.is_contiguous()
                and values.numel() > 0)

    k = Kernels()
    monkeypatch.setattr(_hip, "load", lambda: k)
    monkeypatch.setattr(losses, "_ordinary", ordinary)
    return k


def _problem(dtype=torch.float32, vocab=61, bias=False, seed=1):
    gen = torch.Generator().manual_seed(seed)
    hidden = torch.randn(2, 12, 8, generator=gen).to(dtype).requires_grad_()
    head = torch.nn.Linear(8, vocab, bias=bias, dtype=dtype)
    with torch.no_grad():
        for p in head.parameters():
            p.copy_(torch.randn(p.shape, generator=gen) * 0.4)
    labels = torch.randint(0, vocab, (2, 12), generator=gen)
    labels[:, :3] = IGNORE
    return hidden, head, labels


def _loss(hidden, head, labels, chunk=10):
    return ab.causal_lm_loss(hidden, head, labels, chunk_tokens=chunk)


def _whole(hidden, head, labels):
    """The same loss in plain torch operations."""
    return F.cross_entropy(head(hidden[:, :-1]).flatten(0, 1).float(), labels[:, 1:].flatten(), ignore_index=IGNORE)


def _close(got, want, rel=1e-5):
    return all((a - b).norm() <= rel * b.norm() for a, b in zip(got, want, strict=True))


@pytest.mark.parametrize("chunk", [10, 100])
@pytest.mark.parametrize("vocab", [61, 1 << 14])   # the hidden gradient by torch's product, by the split one's rule
@pytest.mark.parametrize("frozen", [False, True])
def test_backward_under_autocast_keeps_the_forwards_types(kernels, vocab, chunk, frozen):
    hidden, head, labels = _problem(vocab=vocab)
    head.weight.requires_grad_(not frozen)
    inputs = [hidden] if frozen else [hidden, head.weight]
    want = torch.autograd.grad(_whole(hidden, head, labels), inputs)
    loss = _loss(hidden, head, labels, chunk)
    with torch.autocast("cpu", dtype=torch.bfloat16):
        got = torch.autograd.grad(loss, inputs)
    assert "cross_entropy_backward" in kernels.calls
    assert all(g.dtype == torch.float32 for g in got) and _close(got, want)


@pytest.mark.parametrize("counted", [True, False])   # written through torch, or as the update kernels write: no version
def test_a_weight_written_between_the_passes_is_read_as_it_is(kernels, counted):
    hidden, head, labels = _problem()
    loss = _loss(hidden, head, labels)
    new = head.weight.detach() * 40.0   # logits far above the first pass's row maxima
    with torch.no_grad():
        head.weight.copy_(new) if counted else head.weight.data.copy_(new)
    got = torch.autograd.grad(loss, [hidden, head.weight])
    assert "cross_entropy_backward" in kernels.calls
    assert _close(got, torch.autograd.grad(_whole(hidden, head, labels), [hidden, head.weight]))


def test_a_second_backward_needs_the_graph_kept(kernels):
    hidden, head, labels = _problem()
    loss = _loss(hidden, head, labels)
    loss.backward()
    with pytest.raises(RuntimeError, match="backward through the graph a second time"):
        loss.backward()


def test_a_frozen_hidden_state_keeps_the_weights_gradient_of_the_forward_pass(kernels):
    """Without a gradient to the hidden states nothing is computed again: the slices' logits are kept."""
    hidden, head, labels = _problem()
    hidden.requires_grad_(False)
    want = torch.autograd.grad(_whole(hidden, head, labels), head.weight)
    loss = _loss(hidden, head, labels)
    head.weight.data.mul_(3.0)
    assert _close(torch.autograd.grad(loss, head.weight), want)
    assert "cross_entropy_backward" in kernels.calls


class _Watch(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _modes():
    from torch.utils.flop_counter import FlopCounterMode
    return {"function": _Watch, "device": lambda: torch.device("cpu"), "flops": lambda: FlopCounterMode(display=False)}


@pytest.mark.parametrize("head_kind", ["bias", "lambda", "linear"])
@pytest.mark.parametrize("where", ["forward", "backward", "both"])
@pytest.mark.parametrize("mode", ["function", "device", "flops"])
def test_a_mode_around_either_pass(kernels, mode, where, head_kind):
    """The choice between kernels and torch operations is the call's: what a checkpointed slice computes
    again is what it computed first, whatever is active then."""
    hidden, head, labels = _problem(bias=head_kind == "bias")
    project = (lambda x: head(x)) if head_kind == "lambda" else head
    inputs = [hidden, *head.parameters()]
    want = torch.autograd.grad(_whole(hidden, head, labels), inputs)
    from contextlib import nullcontext
    make = _modes()[mode]
    with make() if where != "backward" else nullcontext():
        loss = ab.causal_lm_loss(hidden, project, labels, chunk_tokens=10)
        if where == "both":
            loss.backward()
    with make() if where == "backward" else nullcontext():
        if where != "both":
            loss.backward()
    assert _close([p.grad for p in inputs], want)


def test_a_default_device_around_the_whole_step(kernels):
    hidden, head, labels = _problem(bias=True)
    want = torch.autograd.grad(_whole(hidden, head, labels), [hidden, *head.parameters()])
    torch.set_default_device("cpu")
    try:
        _loss(hidden, head, labels).backward()
    finally:
        torch.set_default_device(None)
    assert _close([hidden.grad, *(p.grad for p in head.parameters())], want)


@pytest.mark.parametrize("bias", [False, True])
def test_a_default_device_does_not_keep_the_kernels_away(kernels, bias):
    """A default device changes where factories put new tensors, and is there for a whole program."""
    hidden, head, labels = _problem(bias=bias)
    torch.set_default_device("cpu")
    try:
        _loss(hidden, head, labels).backward()
        assert kernels.calls.count("cross_entropy_backward") == 3
        kernels.calls.clear()
        with torch.no_grad():
            _loss(hidden, head, labels)
        assert kernels.calls == ["cross_entropy"] * 3
        kernels.calls.clear()
        with _Watch():
            _loss(hidden, head, labels).backward()
        assert not kernels.calls
    finally:
        torch.set_default_device(None)


@pytest.mark.parametrize("head_kind", ["bias", "linear", "frozen"])
def test_batched_gradients(kernels, head_kind):
    """is_grads_batched: the backward pass runs under vmap, its incoming gradient a batch."""
    hidden, head, labels = _problem(bias=head_kind == "bias")
    hidden.requires_grad_(head_kind != "frozen")
    inputs = [x for x in (hidden, *head.parameters()) if x.requires_grad]
    seeds = torch.tensor([0.0, 1.0, -0.3])
    want = torch.autograd.grad(_whole(hidden, head, labels), inputs)
    got = torch.autograd.grad(_loss(hidden, head, labels), inputs, seeds, is_grads_batched=True)
    for g, w in zip(got, want, strict=True):
        assert _close(list(g[1:]), [seeds[1] * w, seeds[2] * w]) and not g[0].any()
    loss = _loss(hidden, head, labels)
    for g, b in zip(got, torch.func.vmap(lambda seed: torch.autograd.grad(loss, inputs, seed))(seeds), strict=True):
        assert torch.allclose(g, b, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("head_kind", ["bias", "linear"])
def test_vectorized_jacobians_and_second_derivatives(kernels, head_kind):
    hidden, head, labels = _problem(bias=head_kind == "bias")
    jacobian = torch.autograd.functional.jacobian(lambda h: _loss(h, head, labels), hidden.detach(), vectorize=True)
    assert _close([jacobian], torch.autograd.grad(_whole(hidden, head, labels), hidden))
    inputs = [hidden, head.weight]

    def second(loss):
        first = torch.autograd.grad(loss, inputs, torch.tensor(0.7), create_graph=True)
        return torch.autograd.grad(sum(g.square().sum() for g in first), inputs)

    assert _close(second(_loss(hidden, head, labels)), second(_whole(hidden, head, labels)), 1e-4)


def test_operations_watched_in_the_backward_pass_are_torchs(kernels):
    from torch.utils.flop_counter import FlopCounterMode
    hidden, head, labels = _problem(torch.bfloat16, vocab=1 << 14)
    inputs = [hidden, head.weight]
    want = torch.autograd.grad(_whole(hidden, head, labels), inputs)
    loss = _loss(hidden, head, labels)
    with FlopCounterMode(display=False) as count:
        got = torch.autograd.grad(loss, inputs)
    assert count.get_total_flops() == 3 * 2 * 24 * 8 * (1 << 14) and "matmul" not in kernels.calls
    assert _close(got, want, 2.0 ** -7)   # the logits' gradient and the result rounded to BF16


def test_a_target_outside_the_vocabulary_has_no_gradient_in_torch_operations_either():
    logits = torch.randn(5, 9, generator=torch.Generator().manual_seed(2), requires_grad=True)
    target = torch.tensor([3, 9, IGNORE, -1, 8])
    grad = losses._logits_gradient(logits, target, IGNORE, torch.tensor(0.0))
    assert grad[[1, 3]].isnan().all() and not grad[[0, 2, 4]].any()
    good = [0, 2, 4]
    loss = F.cross_entropy(logits[good], target[good], ignore_index=IGNORE, reduction="sum")
    want = torch.autograd.grad(loss, logits)[0][good]
    assert torch.allclose(losses._logits_gradient(logits, target, IGNORE, torch.tensor(1.0))[good], want, atol=1e-6)


class _Library:
    """The loaded library where no call may reach it."""

    def __getattr__(self, name):
        raise AssertionError(f"{name} was called")


def test_operands_the_kernels_cannot_take_are_refused():
    """Types, shapes, strides and devices are checked before an address is passed on."""
    k = object.__new__(_hip.HipKernels)
    k._lib = _Library()
    bf16 = dict(dtype=torch.bfloat16)

    a, b, out = torch.zeros(4, 16, **bf16), torch.zeros(16, 8, **bf16), torch.zeros(4, 8, **bf16)
    for wrong in ((a.float(), b, out), (a, b.float(), out), (a, b, out.float()), (a, b, out[:3]), (a, b[:8], out),
                  (a, b, torch.zeros(8, 4, **bf16).t()), (a.t().contiguous().t(), b, out), (a, b, out.to("meta"))):
        with pytest.raises(ValueError, match="must be contiguous"):
            k.matmul(*wrong)

    x, t = torch.zeros(4, 9), torch.zeros(4, dtype=torch.int64)
    for wrong in ((x.half(), t), (x.t().contiguous().t(), t), (x, t.int()), (x, t[:3]), (x, t.to("meta")),
                  (x, torch.zeros(8, dtype=torch.int64)[::2])):
        with pytest.raises(ValueError, match="must be contiguous"):
            k.cross_entropy(*wrong, IGNORE)

    stats, gout = torch.zeros(4, 2), torch.zeros(())
    for wrong in ((x, t, stats[:3], gout, None), (x, t, stats.double(), gout, None), (x, t, stats, gout.double(), None),
                  (x, t, stats, gout[None], None), (x, t, stats, gout, x.bfloat16()), (x, t, stats, gout, x[:, :8]),
                  (x, t.int(), stats, gout, None), (x.half(), t, stats, gout, None), (x, t, stats, gout.to("meta"), None)):
        logits, target, s, g, o = wrong
        with pytest.raises(ValueError, match="must be contiguous"):
            k.cross_entropy_backward(logits, target, IGNORE, s, g, o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_many_short_rows_take_torch_operations(kernels, dtype):
    """Both sides of each line of the two rules: a slice's own kernels, and a bare Linear head's."""
    def slice_taken(rows, vocab):
        return losses._kernels_apply(torch.empty(rows, vocab, dtype=dtype), torch.empty(rows, dtype=torch.int64))

    def head_taken(rows, vocab, chunk):
        head = torch.nn.Linear(2, vocab, bias=False, dtype=dtype)
        return losses._head_applies(head, torch.empty(rows, 2, dtype=dtype), torch.empty(rows, dtype=torch.int64), chunk)

    few, line = losses._SLICE_RULE[0], losses._SLICE_RULE[1][dtype]
    assert slice_taken(few, 1) and slice_taken(few, line) and slice_taken(few + 1, line)
    assert not slice_taken(few + 1, line - 1) and not slice_taken(4 * few, 1)
    few, line = losses._HEAD_RULE[0], losses._HEAD_RULE[1][dtype]
    assert head_taken(few, 2, 2 * few) and head_taken(few + 1, line, 2 * few) and head_taken(4 * few, 2, few)
    assert not head_taken(few + 1, line - 1, 2 * few)
    hidden = torch.randn(1, few + 3, 2).to(dtype).requires_grad_()
    head = torch.nn.Linear(2, 3, bias=False, dtype=dtype)
    labels = torch.randint(0, 3, (1, few + 3))
    for chunk, calls in ((few, True), (few + 3, False)):
        kernels.calls.clear()
        loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=chunk)
        assert bool(kernels.calls) == calls
        got = torch.autograd.grad(loss, [hidden, head.weight])
        tol = 1e-4 if dtype == torch.float32 else 2.0 ** -6   # FP32 sums of 65539 rows; BF16 logits and gradients
        assert _close(got, torch.autograd.grad(_whole(hidden, head, labels), [hidden, head.weight]), tol)


def test_which_products_are_worth_splitting(kernels):
    def split(m, n, k):
        kernels.calls.clear()
        a, b, out = (torch.zeros(1, dtype=torch.bfloat16).expand(shape) for shape in ((m, k), (k, n), (m, n)))
        kernels.matmul = lambda *x: kernels.calls.append("matmul")
        try:
            losses._matmul_into(out, a, b)
        except RuntimeError:   # torch's product refuses an expanded result
            pass
        return bool(kernels.calls)

    assert split(4096, 1024, 1 << 15) and split(1024, 4096, 1 << 15) and split(4096, 64, 1 << 15)
    assert not split(4104, 64, 1 << 15) and not split(4096, 1028, 1 << 15)
    assert split(2048, 1024, 1 << 14) and split(4096, 512, (1 << 15) - 8)
    assert not split(2048, 1028, 1 << 14) and not split(4096, 516, (1 << 15) - 8) and not split(8, 64, (1 << 14) - 8)
