"""The native per-tensor path of an update (csrc/abh_bind.cpp) on tensors it cannot take, on the CPU."""

import subprocess
import sys
from pathlib import Path

_THROWING = r"""
import ctypes
import sys
import types

import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from adambridge_amd import _hip

with FakeTensorMode():
    fake = torch.empty(2, 8, device="cuda:0")
held = torch._C._functorch._add_batch_dim(fake, 0, torch._C._functorch._vmap_increment_nesting(2, "error"))
assert type(held) is torch.Tensor and held.is_cuda   # Python's own type, on a GPU, without memory
try:
    held.data_ptr()
    sys.exit("this tensor has memory")
except RuntimeError:
    pass
seg = _hip.Segment(n=8)
state = object()
slot = types.SimpleNamespace(submitted=False, plain=True, state=state, bound=state, param=held, step=3, group={},
                             seg_addr=ctypes.addressof(seg), in_place=False, small=None)
array = (ctypes.c_void_p * 1)()
assert _hip.bind().describe([slot], [held], array, 0, 0, False, lambda group: 0) is False
assert slot.step == 3 and array[0] is None and not seg.g
print("whole")
"""


def test_native_host_work_survives_a_tensor_without_memory():
    """An exception of torch's C++ side inside describe() leaves the call to the general path, which raises
    it in Python; it does not end the process."""
    run = subprocess.run([sys.executable, "-c", _THROWING], capture_output=True, text=True, timeout=300,
                         cwd=Path(__file__).resolve().parent.parent)
    assert run.returncode == 0 and run.stdout.strip().endswith("whole"), run.stderr[-2000:]
