"""The library's cross-entropy kernels (csrc/abh_loss.hip) against float64 on the same logits, and
causal_lm_loss where the kernels must not be taken."""

import pytest
import torch
import torch.nn.functional as F

import adambridge_amd as ab
from adambridge_amd import _hip, losses

pytestmark = pytest.mark.gpu
IGNORE = -100


def _case(rows, vocab, dtype, seed=0, scale=4.0):
    gen = torch.Generator("cuda").manual_seed(seed)
    logits = (torch.randn(rows, vocab, generator=gen, device="cuda") * scale).to(dtype)
    target = torch.randint(0, vocab, (rows,), generator=gen, device="cuda")
    target[::3] = IGNORE
    return logits, target


def _exact(logits, target, gout):
    logp = logits.double().log_softmax(1)
    keep = (target != IGNORE).double()
    at = target.clamp(min=0)[:, None]
    terms = -logp.gather(1, at)[:, 0] * keep
    grad = (logp.exp().scatter_add(1, at, -torch.ones_like(at, dtype=torch.float64))) * keep[:, None] * gout
    return terms.sum(), terms, grad


# one value, less than a 16-byte vector, a head and a tail around the vectors (odd rows start off the
# 16-byte boundary), one and several workgroups per row, the largest vocabulary
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,vocab", [(1, 1), (5, 7), (4, 8), (3, 2049), (301, 4099), (2050, 1024), (3, 16389),
                                        (2, 151936), (33, 50257), (1025, 9)])
def test_loss_and_gradient_match_float64(rows, vocab, dtype):
    logits, target = _case(rows, vocab, dtype)
    k = _hip.load()
    gout = torch.tensor(0.37, device="cuda")
    loss, stats = k.cross_entropy(logits, target, IGNORE)
    grad = k.cross_entropy_backward(logits, target, IGNORE, stats, gout)
    want, terms, want_grad = _exact(logits, target, 0.37)
    # the sum of FP32 terms: each off by a few ulp of its log-sum (below 32: 4 x 2^-20), their sum by
    # the roundings of a lane's rows and the tree
    assert abs(loss.item() - want.item()) <= rows * 4 * 2.0 ** -20 + abs(want.item()) * 2.0 ** -20
    # p's relative error: |x - m| <= 48 here, times log2(e), rounded once (2^-24 of it), the exponential and
    # two products: below 48 x 1.45 x 2^-24 + 2^-21 < 2^-17; then the rounding to the logits' type
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    p = (want_grad - torch.zeros_like(want_grad)).abs()
    bound = p * unit + 0.37 * logits.double().softmax(1) * 2.0 ** -17 + 1e-38
    assert ((grad.double() - want_grad).abs() <= bound).all()
    assert not grad[::3].any()   # ignored rows


def test_infinities_nan_and_targets_outside_the_vocabulary():
    k = _hip.load()
    gout = torch.ones((), device="cuda")
    logits = torch.randn(8, 300, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    target = torch.arange(8, device="cuda") + 5
    logits[0, 100:] = -torch.inf
    logits[1] = -torch.inf
    logits[2, 7] = torch.nan
    logits[3, 3] = torch.inf
    logits[4, :200] = torch.finfo(torch.float32).min
    logits[5] = torch.finfo(torch.float32).min
    target[6] = IGNORE
    logits[6, 9] = torch.nan   # an ignored row's NaN reaches its gradient, as in torch's operations
    for r in range(8):
        one, t = logits[r:r + 1].clone().requires_grad_(), target[r:r + 1]
        want = F.cross_entropy(one, t, ignore_index=IGNORE, reduction="sum")
        want.backward()
        loss, stats = k.cross_entropy(one.detach(), t, IGNORE)
        grad = k.cross_entropy_backward(one.detach(), t, IGNORE, stats, gout)
        assert torch.allclose(loss, want.detach(), rtol=2e-6, atol=1e-6, equal_nan=True), r
        assert torch.allclose(grad, one.grad, rtol=1e-5, atol=1e-7, equal_nan=True), r
    for bad in (300, -1):
        assert k.cross_entropy(logits[7:], torch.tensor([bad], device="cuda"), IGNORE)[0].isnan()


def _problem(dtype=torch.bfloat16, vocab=997, seed=1):
    gen = torch.Generator("cuda").manual_seed(seed)
    hidden = torch.randn(2, 40, 64, generator=gen, device="cuda").to(dtype).requires_grad_()
    head = torch.nn.Linear(64, vocab, bias=False, device="cuda", dtype=dtype)
    with torch.no_grad():
        head.weight.normal_(0.0, 0.2, generator=gen)
    labels = torch.randint(0, vocab, (2, 40), generator=gen, device="cuda")
    labels[:, :9] = IGNORE
    return hidden, head, labels


def _grads(hidden, head, labels, **kw):
    hidden.grad = head.weight.grad = None
    loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32)
    loss.backward(**kw)
    return loss.detach(), hidden.grad, head.weight.grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_causal_lm_loss_takes_the_kernels_and_agrees_with_torch(dtype, monkeypatch):
    problem = _problem(dtype)
    calls = []
    k = _hip.load()
    real = k.cross_entropy_backward
    monkeypatch.setattr(k, "cross_entropy_backward", lambda *a, **kw: calls.append(kw) or real(*a, **kw))
    got = _grads(*problem)
    assert len(calls) == 3 and all("out" in kw for kw in calls)   # 80 positions, 32 at a time, a plain head
    with torch.autograd.graph.save_on_cpu():
        moved = _grads(*problem)
    monkeypatch.setattr(losses, "_head_applies", lambda *a: False)
    sliced = _grads(*problem)
    assert len(calls) == 9 and not calls[-1]
    monkeypatch.setattr(losses, "_kernels_apply", lambda *a: False)
    want = _grads(*problem)
    # two roundings of the logits' gradient to BF16 (2^-8 apart at most, at random) before the products
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    for a, b, c, d in zip(got, want, moved, sliced):
        assert (a - b).norm() <= tol * b.norm() and (d - b).norm() <= tol * b.norm() and torch.equal(a, c)


def test_second_derivatives_and_transforms_use_torch_operations(monkeypatch):
    hidden, head, labels = _problem(torch.float32, vocab=61)
    target = torch.zeros(80, dtype=torch.int64, device="cuda")
    logits = head(hidden.reshape(80, 64)).detach().requires_grad_()

    def second():
        loss = losses._slice_loss_sum(logits, target, lambda x: x, IGNORE)
        (g,) = torch.autograd.grad(loss, logits, create_graph=True)
        return g.detach(), torch.autograd.grad(g.square().sum(), logits)[0]

    got = second()
    rows = torch.func.vmap(lambda h: losses._slice_loss_sum(h, target[:40], head, IGNORE))(hidden.detach())
    tangent = torch.func.jvp(lambda x: losses._slice_loss_sum(x, target, lambda y: y, IGNORE), (logits.detach(),),
                             (torch.ones_like(logits),))[1]
    monkeypatch.setattr(losses, "_kernels_apply", lambda *a: False)
    want = second()
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-6)
    each = torch.stack([losses._slice_loss_sum(h, target[:40], head, IGNORE) for h in hidden.detach()])
    assert torch.allclose(rows, each, rtol=1e-5)
    assert abs(tangent.item()) < 1e-2   # a shift of every logit leaves the loss as it is


def test_other_types_and_strides_use_torch_operations():
    target = torch.zeros(4, dtype=torch.int64, device="cuda")
    base = torch.randn(4, 66, device="cuda")
    assert losses._kernels_apply(base, target)
    assert not losses._kernels_apply(base[:, :64], target)                      # strided rows
    assert not losses._kernels_apply(base.half(), target)
    assert not losses._kernels_apply(base, target.int())
    assert not losses._kernels_apply(base.reshape(-1)[1:-65].view(3, 66), target[:3])   # off the 16-byte boundary
    assert not losses._kernels_apply(base.cpu(), target.cpu())
    loss = losses._slice_loss_sum(base.half(), target, lambda x: x, IGNORE)
    assert torch.allclose(loss, F.cross_entropy(base.half().float(), target, reduction="sum"))


@pytest.mark.parametrize("frozen", ["none", "hidden", "weight"])
def test_a_plain_head_matches_float64(frozen, monkeypatch):
    """_HeadLoss's gradients, with either input frozen, a seed gradient and a second derivative."""
    hidden, head, labels = _problem(torch.float32, vocab=301)
    hidden.requires_grad_(frozen != "hidden")
    head.weight.requires_grad_(frozen != "weight")
    inputs = [x for x in (hidden, head.weight) if x.requires_grad]
    assert losses._head_applies(head, hidden.reshape(80, 64), torch.zeros(80, dtype=torch.int64, device="cuda"))
    loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32)
    grads = torch.autograd.grad(loss, inputs, torch.tensor(0.3, device="cuda"))
    h64, w64 = hidden.detach().double().requires_grad_(), head.weight.detach().double().requires_grad_()
    target = torch.full_like(labels, IGNORE)
    target[:, :-1] = labels[:, 1:]
    want = F.cross_entropy((h64.reshape(80, 64) @ w64.T), target.reshape(-1), ignore_index=IGNORE)
    exact = dict(zip(("hidden", "weight"), torch.autograd.grad(want, (h64, w64), torch.tensor(0.3, device="cuda").double())))
    assert torch.allclose(loss.double(), want, rtol=1e-6)
    for g, name in zip(grads, [n for n in ("hidden", "weight") if n != frozen]):
        assert (g.double() - exact[name]).norm() <= 1e-5 * exact[name].norm()   # FP32 sums of 301 terms
    loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32)
    first = torch.autograd.grad(loss, inputs, create_graph=True)
    second = torch.autograd.grad(sum(g.square().sum() for g in first), inputs)
    monkeypatch.setattr(losses, "_head_applies", lambda *a: False)
    monkeypatch.setattr(losses, "_kernels_apply", lambda *a: False)
    loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=80)
    first = torch.autograd.grad(loss, inputs, create_graph=True)
    for a, b in zip(second, torch.autograd.grad(sum(g.square().sum() for g in first), inputs)):
        assert (a - b).norm() <= 1e-4 * b.norm()


def test_heads_that_are_called_as_they_are():
    """Anything but a bare Linear keeps its own call."""
    hidden, head, labels = _problem(torch.bfloat16)
    h, t = hidden.reshape(80, 64), torch.zeros(80, dtype=torch.int64, device="cuda")
    assert losses._head_applies(head, h, t)
    assert not losses._head_applies(lambda x: head(x), h, t)
    assert not losses._head_applies(torch.nn.Linear(64, 9, device="cuda", dtype=torch.bfloat16), h, t)   # a bias
    assert not losses._head_applies(head, h.float(), t) and not losses._head_applies(head, h[::2], t[::2])
    assert not losses._head_applies(head.cpu(), h, t)
    head.cuda()
    handle = head.register_forward_hook(lambda *a: None)
    assert not losses._head_applies(head, h, t)
    handle.remove()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not losses._head_applies(head, h, t)
    head.forward = lambda x: F.linear(x, head.weight)
    assert not losses._head_applies(head, h, t)
    del head.forward
    assert losses._head_applies(head, h, t)
    torch.nn.utils.parametrizations.weight_norm(head)
    assert not losses._head_applies(head, h, t)


# one row, the ends of a tile (256 x 128), a step (64 terms) and a split; rows and columns past a tile
@pytest.mark.parametrize("m,n,k", [(1, 4, 8), (3, 8, 64), (33, 124, 72), (255, 128, 1024), (256, 132, 2056), (257, 4, 4096),
                                   (1024, 896, 16392), (333, 1536, 50264), (2, 260, 151936)])
def test_split_product_matches_float64(m, n, k):
    gen = torch.Generator("cuda").manual_seed(m + n)
    a = torch.randn(m, k, generator=gen, device="cuda").bfloat16()
    b = torch.randn(k, n, generator=gen, device="cuda").bfloat16()
    room = torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device="cuda")
    _hip.load().matmul(a, b, room[1:m + 1])
    want = a.double() @ b.double()
    # one rounding to BF16 (8 significant bits: half a last place is at most 2^-8 of the value), and FP32
    # sums of k products: each of the k additions off by 2^-24 of a partial sum, at most |a| |b| in all
    bound = want.abs() * 2.0 ** -8 + (a.double().abs() @ b.double().abs()) * 2.0 ** -24 * k ** 0.5 + 1e-30
    assert ((room[1:m + 1].double() - want).abs() <= bound).all()
    assert (room[0] == 7).all() and (room[-1] == 7).all()


def test_which_products_are_split(monkeypatch):
    k = _hip.load()
    calls = []
    monkeypatch.setattr(k, "matmul", lambda a, b, out: calls.append(a.shape))
    def try_(m, n, kk, dtype=torch.bfloat16, offset=0):
        calls.clear()
        a = torch.zeros(m * kk + offset, dtype=dtype, device="cuda")[offset:].view(m, kk)
        losses._matmul_into(torch.empty(m, n, dtype=dtype, device="cuda"), a, torch.zeros(kk, n, dtype=dtype, device="cuda"))
        return bool(calls)
    assert try_(8, 64, 1 << 14) and try_(8, 68, 20008)
    assert not try_(8, 64, 8192) and not try_(8, 66, 1 << 14) and not try_(8, 64, 20004)
    assert not try_(8, 64, 1 << 14, torch.float32) and not try_(8, 64, 1 << 14, offset=4)
    assert not try_(2056, 2048, 1 << 14)


@pytest.mark.parametrize("bias", [False, True])
def test_backward_passes_of_other_kinds(bias, monkeypatch):
    """Batched gradients, a pass under autocast, a default device, a step between the forward and the backward
    pass: on the kernels where they apply, the torch operations' results everywhere."""
    hidden, head, labels = _problem(torch.float32, vocab=1 << 14)
    if bias:
        head.bias = torch.nn.Parameter(torch.zeros(1 << 14, device="cuda"))
    seeds = torch.tensor([1.0, -0.3], device="cuda")

    def results(kernels):
        inputs = [hidden, *head.parameters()]
        opt = ab.AdamBridge(head.parameters(), lr=1e-2)
        start = head.weight.detach().clone()
        out = list(torch.autograd.grad(ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32), inputs, seeds,
                                       is_grads_batched=True))
        loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=not bias and kernels):   # torch's products take BF16 there
            out += torch.autograd.grad(loss, inputs)
        torch.set_default_device("cuda")
        try:
            out += torch.autograd.grad(ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32), inputs)
        finally:
            torch.set_default_device(None)
        loss = ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32)
        for p in head.parameters():   # the same update on both sides
            p.grad = torch.randn(p.shape, generator=torch.Generator("cuda").manual_seed(5), device="cuda")
        opt.step()
        out += torch.autograd.grad(loss, inputs)
        with torch.no_grad():
            head.weight.copy_(start)
            head.weight.grad = None
            if bias:
                head.bias.zero_()
                head.bias.grad = None
        return out

    got = results(True)
    monkeypatch.setattr(losses, "_head_applies", lambda *a: False)
    monkeypatch.setattr(losses, "_kernels_apply", lambda *a: False)
    for i, (a, b) in enumerate(zip(got, results(False), strict=True)):
        assert a.dtype == b.dtype == torch.float32 and (a - b).norm() <= 1e-5 * b.norm(), i   # as in the tests above


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [7, 300, 20001])   # the row in values, in vectors with a tail, over several workgroups
def test_a_target_outside_the_vocabulary_has_no_gradient(vocab, dtype):
    """NaN over its whole row, as the loss is, and in no other."""
    logits, target = _case(6, vocab, dtype)
    target[1], target[2], target[4] = vocab, -1, vocab + 5
    k = _hip.load()
    loss, stats = k.cross_entropy(logits, target, IGNORE)
    for gout in (torch.ones((), device="cuda"), torch.zeros((), device="cuda")):
        grad = k.cross_entropy_backward(logits, target, IGNORE, stats, gout)
        same = losses._logits_gradient(logits, target, IGNORE, gout)
        for g in (grad, same):
            assert loss.isnan() and g[[1, 2, 4]].isnan().all() and not g[[0, 3, 5]].isnan().any()


@pytest.mark.parametrize("bias", [False, True])
def test_second_derivatives_with_deterministic_algorithms(bias):
    hidden, head, labels = _problem(torch.float32, vocab=61)
    if bias:
        head.bias = torch.nn.Parameter(torch.zeros(61, device="cuda"))
    inputs = [hidden, head.weight]
    results = []
    for loss_of in (lambda: ab.causal_lm_loss(hidden, head, labels, chunk_tokens=32),
                    lambda: F.cross_entropy(head(hidden[:, :-1]).flatten(0, 1), labels[:, 1:].flatten(), ignore_index=IGNORE)):
        torch.use_deterministic_algorithms(True)
        try:
            first = torch.autograd.grad(loss_of(), inputs, create_graph=True)
            results.append(torch.autograd.grad(sum(g.square().sum() for g in first), inputs))
        finally:
            torch.use_deterministic_algorithms(False)
    for a, b in zip(*results):
        assert (a - b).norm() <= 1e-4 * b.norm()   # as the second derivatives above
