"""The separate FP32 / BF16-moment kernel's lane widths (four elements, two, one) against the oracle, at the
ends of a lane, a workgroup's pass and a tile."""

import itertools

import numpy as np
import pytest
import torch

from hip_cases import run_hip
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# a buffer moved by 1 element allows one-element accesses only, by 2 pairs, by 4 all; one moved
# buffer among aligned ones decides for all
@pytest.mark.parametrize("shift,which", [(0, "all"), (1, "all"), (2, "all"), (4, "all"), (2, "g"), (2, "out"), (1, "p_lo")])
@pytest.mark.parametrize("algo", [O.ADAMW, O.LION])
def test_lane_widths_match_oracle(algo, shift, which):
    rng = np.random.default_rng(shift * 10 + algo)
    cases = []
    for mv, pt, (gt, ot) in itertools.product((O.DT_F32, O.DT_BF16), (O.DT_F32, O.DT_F24),
                                              ((O.DT_BF16, O.DT_BF16), (O.DT_F32, O.DT_F32), (O.DT_F32, O.DT_NONE))):
        for n in (1, 3, 4, 6, 16, 19, 511, 512, 514, 1023, 1028, 4099):
            cases.append(O.make_case(rng, n, algorithm=algo, mv_dtype=mv, p_dtype=pt, g_dtype=gt, out_dtype=ot,
                                     index=len(cases), step=1 + n % 7, offset=int(rng.integers(0, 2**32))))

    def move(i, tensors):
        for k, t in list(tensors.items()):
            if which in ("all", k):
                buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=t.device)
                buf[shift:].copy_(t)
                tensors[k], tensors["_keep" + k] = buf[shift:], buf

    for width in (16, 0):
        for flags in (0, 1):   # 1: out receives the weight from before the update
            want = O.run_many(cases, "oracle", width)
            got = run_hip(cases, width, tensors_hook=move if shift else None, seg_flags=flags)
            for w, g in zip(want, got):
                skip = ("out",) if flags else ()
                bad = [k for k in O.outputs_equal(w, g) if k not in skip]
                assert not bad, (w.n, w.mv_dtype, w.p_dtype, bad)
