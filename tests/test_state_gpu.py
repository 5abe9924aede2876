"""Interleaved states to and from separate arrays on the device (adambridge_pack_state,
adambridge_unpack_state) against the same states in host memory, whose strided-view code is the
oracle here (checked element by element in test_host_cpu.py), byte for byte."""

import numpy as np
import pytest
import torch

import adambridge_amd as ab
from adambridge_amd import precision as P
from adambridge_amd import state as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
KINDS = {"pairs": ("adamw", "bf16", "fp32"), "fp8-records": ("adamw", "fp8", "fp32"),
         "lion-records": ("lion", "bf16", "fp32"), "f32-records": ("adamw", "fp32", "fp32"),
         "f24-records": ("adamw", "bf16", "fp24"), "lion-f24-records": ("lion", "bf16", "fp24"),
         "fp8-f24-records": ("adamw", "fp8", "fp24"), "lion-f32-records": ("lion", "fp32", "fp32"),
         "lion-fp8-records": ("lion", "fp8", "fp32"), "f24-f32-records": ("adamw", "fp32", "fp24"),
         "lion-f24-f32-records": ("lion", "fp32", "fp24"), "lion-fp8-f24-records": ("lion", "fp8", "fp24")}
# ends of a lane's 4 or 8 elements, of a pair, a block, a record and a workgroup's share
SIZES = [1, 2, 3, 4, 5, 7, 8, 127, 128, 129, 255, 256, 257, 1023, 2049, 70001]


def _values(n, seed):
    """(master, m, v) in FP32 with special values among them; v a square of 8-bit numbers, so that its root
    is exact on any host."""
    rng = np.random.default_rng((n, seed))
    p = rng.standard_normal(n).astype(np.float32)
    m = (rng.standard_normal(n) * 10.0 ** rng.integers(-8, 1, n)).astype(np.float32)
    u = rng.integers(1, 256, n).astype(np.float32) * np.float32(2.0) ** rng.integers(-20, 0, n).astype(np.float32)
    v = u * u
    for a, specials in ((p, [0.0, -0.0, np.nan, np.inf]), (m, [0.0, -0.0, np.nan, -np.inf]), (v, [0.0, np.nan])):
        for x in specials:
            if n > 4:
                a[rng.integers(0, n)] = x
    return torch.from_numpy(p), torch.from_numpy(m), torch.from_numpy(v)


def _state(layout, n, device):
    return S._INTERLEAVED[layout](n, device)


def _buffers(state):
    return [state.current.reshape(-1).view(torch.uint8).cpu()] + [s.cpu() for s in state.scales.values()]


def _same(a, b):
    if isinstance(a, dict):
        return a.keys() == b.keys() and all(_same(a[k], b[k]) for k in a)
    if isinstance(a, torch.Tensor):
        return torch.equal(a.cpu().reshape(-1).view(torch.uint8), b.cpu().reshape(-1).view(torch.uint8))
    return a == b


def _on(store, offset=0):
    """``store`` on the device, each of its tensors ``offset`` values into a larger allocation."""
    def move(t):
        big = torch.zeros(t.numel() + offset, dtype=torch.uint8 if t.element_size() == 1 else t.dtype, device=DEV)
        big[offset:] = t.view(big.dtype) if t.element_size() == 1 else t
        return big[offset:].view(t.dtype)
    if isinstance(store, P.FP8Store):
        return P.FP8Store.wrap(move(store.q), move(store.scale), store.numel, store.role, store.block)
    return type(store).wrap(move(store.data))


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "one value off"])
@pytest.mark.parametrize("layout", sorted(KINDS))
def test_pack_and_unpack_match_the_host(layout, offset):
    algo, precision, master = KINDS[layout]
    for n in SIZES:
        p, m, v = _values(n, 0)
        moments = {"m": P.make_store(precision, n, "m", init=m)}
        if algo == "adamw":
            moments["v"] = P.make_store(precision, n, "v", init=v)
        host, dev = _state(layout, n, "cpu"), _state(layout, n, DEV)
        saved = p if master == "fp32" else P.FP24Store(n, init=p).state_dict()
        on_device = torch.cat([torch.zeros(offset), p]).to(DEV)[offset:] if master == "fp32" else \
            {"precision": "fp24", "hi": torch.cat([torch.zeros(offset, dtype=torch.bfloat16), saved["hi"]]).to(DEV)[offset:],
             "lo": torch.cat([torch.zeros(offset, dtype=torch.uint8), saved["lo"]]).to(DEV)[offset:]}
        host.load(master=saved, moments=moments)
        dev.load(master=on_device, moments={r: _on(s, offset) for r, s in moments.items()})
        for a, b in zip(_buffers(host), _buffers(dev)):
            assert _same(a, b), (n, "packed")
        assert _same(host.export(), dev.export()), (n, "unpacked")
        for role in host.roles:
            assert _same(host.moment(role).state_dict(), dev.moment(role).state_dict()), (n, role)
        # a column at a time, the rest kept
        q, m2, _ = _values(n, 1)
        store = P.make_store(precision, n, "m", init=m2)
        host.load(master=q)
        dev.load(master=q.to(DEV))
        host.load(moments={"m": store})
        dev.load(moments={"m": _on(store)})
        for a, b in zip(_buffers(host), _buffers(dev)):
            assert _same(a, b), (n, "one column")


@pytest.mark.parametrize("source", ["fp32", "bf16", "fp8"])
@pytest.mark.parametrize("layout", sorted(KINDS))
def test_packing_converts_as_the_stores_do(layout, source):
    """Moments of another precision, a bf16 master, stores of another role or block size."""
    algo, precision, master = KINDS[layout]
    for n in (3, 257, 4099):
        p, m, v = _values(n, 2)
        # NaN payloads: a NaN code's as FP32 is the decoder's own (IEEE 754 leaves it open), and a store of the
        # layout's own format is copied with whatever it holds
        if source in ("fp8", precision):
            m, v = m.nan_to_num(1.0), v.nan_to_num(1.0)
        roles = ("m", "v") if algo == "adamw" else ("m",)
        stores = {r: P.make_store(source, n, r, init={"m": m, "v": v}[r]) for r in roles}
        # the values in the layout's own format, encoded by adambridge_convert (test_convert_gpu.py), then
        # packed as they are (the test above)
        native = {r: P.make_store(precision, n, r, init=s.to_fp32().to(DEV)) for r, s in stores.items()}
        want, got = _state(layout, n, DEV), _state(layout, n, DEV)
        want.load(master=p.bfloat16().float().to(DEV), moments=native)
        got.load(master=p.bfloat16().to(DEV), moments={r: _on(s) for r, s in stores.items()})
        keep = ~p.isnan()   # a BF16 NaN is copied bit for bit into FP24, an FP32 one quietened
        assert _same(want.master_fp32().cpu()[keep], got.master_fp32().cpu()[keep])
        for role in roles:
            assert _same(want.moment(role).state_dict(), got.moment(role).state_dict()), (n, role)
        odd = P.FP8Store(n, "m", init=m.nan_to_num(1.0), block=64)
        got.load(moments={"m": odd})
        assert _same(got.moment("m").state_dict(),
                     P.make_store(precision, n, "m", init=odd.to_fp32().to(DEV)).state_dict()), n


@pytest.mark.parametrize("precision,master", [("bf16", "fp32"), ("fp8", "fp24"), ("fp32", "fp32")])
def test_loading_keeps_the_state_in_place(precision, master):
    """load_state_dict on an optimizer that has its state writes into it, and gives what a new optimizer
    gets; its own checkpoint leaves every byte."""
    def build(seed):
        gen = torch.Generator(DEV).manual_seed(seed)
        params = [torch.nn.Parameter(torch.randn(k, generator=gen, device=DEV).bfloat16()) for k in (70, 4099, 256)]
        for p in params:
            p.grad = torch.randn(p.shape, generator=gen, device=DEV).bfloat16()
        opt = ab.AdamBridge(params, precision=precision, master_precision=master)
        for _ in range(2):
            opt.step()
        return opt
    donor, opt = build(1), build(2)
    saved = donor.state_dict()
    at = [s.state.current.data_ptr() for s in opt._ordered]
    opt.load_state_dict(saved)
    assert [s.state.current.data_ptr() for s in opt._ordered] == at
    for a, b in zip(donor._ordered, opt._ordered):
        assert b.step == a.step
        assert all(_same(x, y) for x, y in zip(_buffers(a.state), _buffers(b.state)))
    before = [_buffers(s.state) for s in opt._ordered]
    opt.load_state_dict(opt.state_dict())
    for s, b in zip(opt._ordered, before):
        assert all(_same(x, y) for x, y in zip(_buffers(s.state), b))
    assert all(saved["state"][i]["master"] is not None for i in range(3))


def test_state_argument_codes():
    """Arguments the library refuses, before anything is launched."""
    from adambridge_amd import _hip
    lib = _hip.open_library()
    buf = torch.zeros(4096, dtype=torch.uint8, device=DEV)
    at = buf.data_ptr()

    def call(pack, n=8, layout=_hip.DT_PACKED, data=at, **kw):
        fn = lib.adambridge_pack_state if pack else lib.adambridge_unpack_state
        return fn(_hip.State(data, None, None, n, layout, 0), _hip.Arrays(**kw))

    assert call(True, n=-1) == -1 and call(True, n=0) == 0 and call(True) == 0
    assert call(True, layout=_hip.DT_F32) == -13 and call(True, data=None) == -2
    assert call(True, data=at + 8) < 0
    assert call(False, p=at + 1024, p_dtype=_hip.DT_BF16) == -13
    assert call(True, p=at + 1024, p_dtype=_hip.DT_F24) == -2
    assert call(True, m=at + 1024, mv_dtype=_hip.DT_FP8) == -7
    assert call(False, m=at + 1024, mv_dtype=_hip.DT_F32) == -4
    assert call(True, layout=_hip.DT_PACKED_LION, v=at + 1024, mv_dtype=_hip.DT_BF16) == -4
    assert call(True, layout=_hip.DT_PACKED8, m=at + 1024, m_scale=at, mv_dtype=_hip.DT_FP8) == -7
    assert call(True, p=at + 1026, p_dtype=_hip.DT_F32) < 0
    assert not buf.any()
