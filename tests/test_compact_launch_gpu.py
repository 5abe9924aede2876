"""Launches whose segment descriptors travel in the short form in the kernel arguments, and the calls beside
them that must not take it, against the oracle (bit-exact)."""

import ctypes

import numpy as np
import pytest
import torch

from adambridge_amd import _hip
from hip_cases import (run_hip_f24_records, run_hip_f32_records, run_hip_lion_f32_records, run_hip_lion_records,
                       run_hip_packed, run_hip_records)
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LAYOUTS = {"pairs": (run_hip_packed, dict(mv_dtype=O.DT_BF16)),
           "lion": (run_hip_lion_records, dict(algorithm=O.LION, mv_dtype=O.DT_BF16)),
           "f32": (run_hip_f32_records, dict(mv_dtype=O.DT_F32)),
           "lion-f32": (run_hip_lion_f32_records, dict(algorithm=O.LION, mv_dtype=O.DT_F32)),
           "f24": (run_hip_f24_records, dict(mv_dtype=O.DT_BF16, p_dtype=O.DT_F24)),
           "fp8": (run_hip_records, dict(mv_dtype=O.DT_FP8)),
           "fp8-f24": (run_hip_records, dict(mv_dtype=O.DT_FP8, p_dtype=O.DT_F24)),
           "lion-fp8": (run_hip_records, dict(algorithm=O.LION, mv_dtype=O.DT_FP8)),
           "lion-f24-f32": (run_hip_f24_records, dict(algorithm=O.LION, mv_dtype=O.DT_F32, p_dtype=O.DT_F24))}


# 7 fit as full descriptors, 8 to 78 (FP8: 58) in the short form, up to 312 (232) in several such launches,
# more need a table, and so does one segment with other coefficients among 20; several tiles and scalar tails
@pytest.mark.parametrize("count,odd", [(7, None), (8, None), (78, None), (79, None), (157, None), (312, None), (58, None), (59, None), (232, None),
                                       (313, None), (20, 0), (20, 19)])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_segment_counts_match_oracle(layout, count, odd):
    run, kw = LAYOUTS[layout]
    rng = np.random.default_rng(count)
    sizes = [1, 127, 128, 129, 40001, 255, 5000] + [int(n) for n in rng.integers(1, 6000, count)]
    cases = [O.make_case(rng, sizes[k], index=7 * k, offset=128 * int(rng.integers(0, 2**25)), step=4 if k == odd else 3,
                         stochastic=k % 3 != 0, **kw) for k in range(count)]
    for width in (16, 0):
        for flags in (0, 1):   # 1: out receives the weight from before the update
            want = O.run_many(cases, "oracle", width)
            got = run(cases, width, seg_flags=flags)
            for w, g in zip(want, got):
                bad = [k for k in O.outputs_equal(w, g) if not (flags and k == "out")]
                assert not bad, (w.n, w.index, width, bad)


def test_captured_noalloc_call_matches_multi_step():
    """The allocation-free call of 100 interleaved segments (two launches), captured: each replay applies the
    same update as an eager adambridge_multi_step on a copy of the state."""
    rng = np.random.default_rng(5)
    kernels = _hip.load()
    group = _hip.Group(lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01, seed=3, stochastic=1)
    sides = [[], []]
    for k in range(100):
        n = int(rng.integers(1, 5000))
        state = torch.from_numpy(rng.normal(0, 1e-3, (-(-n // 2), 4)).astype(np.float32)).cuda()
        state.view(torch.int32)[:, 3].bitwise_and_(0x3FFF3FFF)   # v: two BF16 numbers, finite and positive
        state.view(torch.int32)[:, 2].bitwise_and_(-0x40004001)  # m: finite
        g = torch.from_numpy(rng.normal(0, 1e-3, n).astype(np.float32)).cuda()
        for side in sides:
            s, out = state.clone(), torch.zeros(n, dtype=torch.bfloat16, device="cuda")
            side.append((_hip.Segment(p=s.data_ptr(), g=g.data_ptr(), out=out.data_ptr(), group=ctypes.pointer(group), n=n,
                                      step=2, index=k, g_dtype=O.DT_F32, mv_dtype=O.DT_BF16, out_dtype=O.DT_BF16,
                                      p_dtype=_hip.DT_PACKED), s, out, g))
    eager, captured = [kernels.segment_array([ctypes.pointer(e[0]) for e in side]) for side in sides]
    kernels.set_stream(torch.cuda.current_stream())
    kernels.multi_step(None, eager)
    kernels.multi_step_noalloc(torch.cuda.current_stream(), captured)
    graph, other = torch.cuda.CUDAGraph(), torch.zeros(64, device="cuda")
    with torch.cuda.graph(graph):
        kernels.multi_step_noalloc(torch.cuda.current_stream(), captured)
    for replay in range(3):
        graph.replay()
        torch.cuda.synchronize()
        kernels.set_stream(torch.cuda.current_stream())
        kernels.multi_step(None, eager)
        other.add_(1.0)
        torch.cuda.synchronize()
        for (_, s, out, _), (_, t, out2, _) in zip(*sides):
            assert torch.equal(s.view(torch.int32), t.view(torch.int32)) and torch.equal(out, out2), replay
    assert other[0].item() == 3
