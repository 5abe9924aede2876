"""The native per-tensor path of an update (UpdateEngine.update_plain, csrc/abh_bind.cpp) against the general
one, bit for bit, and the calls it leaves to it."""

import pytest
import torch

import adambridge_amd as ab
from adambridge_amd.engine import UpdateEngine

pytestmark = pytest.mark.gpu
SHAPES = [(33, 65), (7,), (128,), (300, 129), (1,), (70001,)]


def _params(dtype, seed=0):
    gen = torch.Generator("cuda").manual_seed(seed)
    return [torch.nn.Parameter(torch.randn(s, generator=gen, device="cuda").to(dtype)) for s in SHAPES]


def _run(dtype, steps=4, grad_dtype=None, skip=(), strided=(), **kw):
    """Parameters, masters and step counts after ``steps`` steps, two groups with changing learning rates;
    parameter k has no gradient in step k % 3 of ``skip``."""
    params = _params(dtype)
    cls = ab.LionBridge if kw.pop("lion", False) else ab.AdamBridge
    opt = cls([{"params": params[:3], "lr": 1e-2}, {"params": params[3:]}], lr=1e-3, small_param_threshold=100, **kw)
    gen = torch.Generator("cuda").manual_seed(9)
    for t in range(steps):
        opt.param_groups[1]["lr"] = 1e-3 / (t + 1)
        for k, p in enumerate(params):
            g = torch.randn(p.shape, generator=gen, device="cuda").to(grad_dtype or dtype)
            if k in strided and g.dim() == 2:
                g = g.t().contiguous().t()
            p.grad = None if k in skip and t % 3 == k % 3 else g
        opt.step()
    opt.flush()
    return [p.detach().clone() for p in params], [m.clone() for m in opt.master_params()], [s.step for s in opt._ordered]


@pytest.mark.parametrize("kw", [
    dict(dtype=torch.float32), dict(dtype=torch.float32, precision="bf16", skip=(1, 4)),
    dict(dtype=torch.bfloat16), dict(dtype=torch.bfloat16, precision="fp8", master_precision="fp24"),
    dict(dtype=torch.bfloat16, precision="bf16", lion=True, skip=(0,)),
    dict(dtype=torch.bfloat16, precision="bf16", delay_updates=True, skip=(2,)),
    dict(dtype=torch.bfloat16, precision="bf16", strided=(0, 3)),
    dict(dtype=torch.float32, precision="bf16", state_layout="separate", overlap_writeback=False),
], ids=str)
def test_native_and_general_paths_give_the_same_bytes(kw, monkeypatch):
    taken = []
    real = UpdateEngine.update_plain
    monkeypatch.setattr(UpdateEngine, "update_plain", lambda *a, **k: taken.append(real(*a, **k)) or taken[-1])
    native = _run(**kw)
    assert any(taken) != bool(kw.get("strided")) and not taken[0]   # the first call builds the states
    monkeypatch.setattr(UpdateEngine, "update_plain", lambda *a, **k: False)
    general = _run(**kw)
    for a, b in zip(native[0] + native[1], general[0] + general[1]):
        assert torch.equal(a, b)
    assert native[2] == general[2]


def test_what_the_native_path_leaves_to_the_general_one():
    """describe() refuses, with step counts and segments as they were."""
    def case(dtype=torch.bfloat16, **kw):
        params = _params(dtype)
        opt = ab.AdamBridge(params, precision="bf16", **kw)
        grads = [torch.randn_like(p) for p in params]
        for p, g in zip(params, grads):
            p.grad = g
        opt.step()
        return opt, opt._engine, list(opt._ordered), grads

    for kw in (dict(double_buffer=True), dict(update_stream="side"), dict(autotune=True)):
        opt, engine, slots, grads = case(**kw)
        assert not engine.update_plain(slots, grads) and [s.step for s in slots] == [1] * len(slots)
    opt, engine, slots, grads = case(overlap_writeback=False)
    assert not engine.update_plain(slots, grads, hooked=True) and engine.update_plain(slots, grads)
    opt, engine, slots, grads = case()
    for k, bad in ((0, grads[0].t().contiguous().t()), (1, grads[1].half()), (2, grads[2][:100]), (3, grads[3].cpu()),
                   (0, torch.randn(33, 130, device="cuda").bfloat16()[:, ::2])):
        assert not engine.update_plain(slots, grads[:k] + [bad] + grads[k + 1:])
    slots[2].submitted = True
    assert not engine.update_plain(slots, grads)
    slots[2].submitted = False
    assert [s.step for s in slots] == [1] * len(slots)
    # a group that cannot be read, and a launch that fails: nothing counted, the error surfaces
    wd = opt.param_groups[0].pop("weight_decay")
    with pytest.raises(RuntimeError, match="adambridge update failed"):
        opt.step()
    opt.param_groups[0]["weight_decay"] = wd
    kernels = engine.kernels
    engine.kernels = type("K", (), {"set_stream": kernels.set_stream,
                                    "multi_step": staticmethod(lambda *a: (_ for _ in ()).throw(RuntimeError("no")))})
    with pytest.raises(RuntimeError, match="adambridge update failed: no"):
        opt.step()
    engine.kernels = kernels
    assert [s.step for s in slots] == [1] * len(slots)
    opt.step()
    assert [s.step for s in slots] == [2] * len(slots)


def test_a_second_gradient_before_the_step_is_refused():
    params = _params(torch.bfloat16)
    opt = ab.AdamBridge(params, precision="bf16", release_grads=False, small_param_threshold=0).attach_hooks()
    for _ in range(2):
        for p in params:
            p.grad = None
        sum(p.float().square().sum() for p in params).backward()
        opt.step_sync()
    sum(p.float().square().sum() for p in params).backward()
    with pytest.raises(RuntimeError, match="second gradient"):
        sum(p.float().square().sum() for p in params).backward()
