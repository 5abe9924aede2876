"""What an interleaved state hands to the packing kernel, on the CPU (the kernel itself is not called)."""

import pytest
import torch

from adambridge_amd.precision import BF16Store, FP8Store, FP32Store
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
