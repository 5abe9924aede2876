"""What an interleaved state hands to the packing kernel, on the CPU (the kernel itself is not called)."""

import pytest
import torch

from adambridge_amd.optimizer import _CheckpointReader
from adambridge_amd.precision import BF16Store, FP8Store, FP32Store, store_from_state_dict
from adambridge_amd.state import AdamRecordState, F24RecordState, PairState


@pytest.mark.parametrize("cls", [PairState, AdamRecordState, F24RecordState])
@pytest.mark.parametrize("size", [0, 255, 299, 301, 512])
def test_arrays_of_another_size_are_refused_before_the_kernel_reads_them(cls, size, monkeypatch):
    state = cls(300, "cpu")
    moved = []
    monkeypatch.setattr(state, "_move", lambda arrays, pack: moved.append(pack))
    for store in (FP32Store(size), BF16Store(size), FP8Store(size, "m"), FP8Store(size, "v")):
        with pytest.raises(ValueError, match="300"):
            state._packed(None, {"m": store})
        with pytest.raises(ValueError, match="300"):
            state._packed(None, {"m": FP32Store(300), "v": store})
    for master in (torch.zeros(size), torch.zeros(size, dtype=torch.bfloat16), FP32Store(size).state_dict(),
                   {"precision": "fp24", "hi": torch.zeros(size, dtype=torch.bfloat16), "lo": torch.zeros(300, dtype=torch.uint8)},
                   {"precision": "fp24", "hi": torch.zeros(300, dtype=torch.bfloat16), "lo": torch.zeros(size, dtype=torch.uint8)}):
        with pytest.raises(ValueError, match="300"):
            state._packed(master, {})
    assert not moved
    state._packed(torch.zeros(300), {"m": FP32Store(300), "v": BF16Store(300)})
    assert moved == [True, True]


class _Sub(torch.Tensor):
    """A subclass may hold its values elsewhere than in memory of its own."""


@pytest.mark.parametrize("kind", ["negated", "subclass"])
@pytest.mark.parametrize("form", ["fp32", "bf16", "fp8", "tensor"])
def test_a_checkpoints_tensors_stand_in_a_store_only_as_memory_holding_their_values(form, kind):
    """The packing kernel reads the memory at a store's address."""
    x = torch.randn(300, generator=torch.Generator().manual_seed(1)).square()

    def shown(t):   # the values of t, not in its memory
        return torch._neg_view(t.neg()) if kind == "negated" else t.as_subclass(_Sub)

    if form == "tensor":
        got, want = _CheckpointReader.moment(shown(x), 300, "v", "bf16", x.device, borrow=True), FP32Store(300, init=x)
    else:
        want = {"fp32": FP32Store, "bf16": BF16Store}[form](300, init=x) if form != "fp8" else FP8Store(300, "v", init=x)
        saved = want.state_dict()
        name = "scale" if form == "fp8" else "data"
        saved[name] = shown(saved[name])
        got = store_from_state_dict(saved, 300, "v", device="cpu", borrow=True)
    assert got.precision == want.precision
    for a, b in zip(got.tensors, want.tensors, strict=True):
        assert type(a) is torch.Tensor and not a.is_neg() and torch.equal(a.view(torch.uint8), b.view(torch.uint8))
