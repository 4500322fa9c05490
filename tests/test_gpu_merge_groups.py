"""The merge of few segments takes 512 / head size heads of a row per wave, 8 channels per lane: head counts that fill
the last wave's groups, leave some idle and need several waves, output rows at every alignment its stores tell apart.

Tolerance: fp32 sums of at most 16 terms, then one rounding to bf16 (2^-8 of the value), doubled; the rotation sums
head size terms, so its rows are compared at their largest value."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import i32, to_f32
from test_gpu_merge import _partials

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("off", [0, 2, 1], ids=["aligned16", "aligned4", "aligned2"])
@pytest.mark.parametrize("hs,nq", [(64, 8), (64, 17), (128, 4), (128, 9), (256, 3), (512, 2)])
def test_head_groups(device, hs, nq, off):
    import torch

    from vllm_quantpack import _hip
    from vllm_quantpack.attention import rht
    S = 9                                             # one full batch of 8 and a remainder
    rng = np.random.default_rng(hs * 7 + nq + off)
    lens = [(1, 1), (4, 9 * 32 * 5 + 3), (2, 200)]
    acc, m, l_, want, want_lse = _partials(rng, lens, nq, S, hs)
    rows = acc.shape[0]
    so, sm, ss = (torch.from_numpy(x).to(device) for x in (acc, m, l_))
    cu_t = i32(np.concatenate(([0], np.cumsum([T for T, _ in lens]))), device)
    used_t = i32([n for _, n in lens], device)
    rotated = (O.rht(want, inverse=True) / hs).astype(np.float32)
    for signs, ref in ((None, want), (rht.signs(hs, device), rotated)):
        wide = torch.full((rows, nq, hs + 8), float("nan"), dtype=torch.bfloat16, device=device)
        out = wide[:, :, off:hs + off]
        lse = torch.full((rows, nq), float("nan"), dtype=torch.float32, device=device)
        args = _hip.MergeArgs(so.data_ptr(), _hip.I64x3(*so.stride()[:3]), sm.data_ptr(), ss.data_ptr(),
                              _hip.I64x2(sm.stride(0), sm.stride(1)), cu_t.data_ptr(), used_t.data_ptr(), len(lens),
                              rows, nq, hs, S, out.data_ptr(), _hip.I64x2(out.stride(0), out.stride(1)),
                              lse.data_ptr(), _hip.I64x2(lse.stride(0), lse.stride(1)), _hip.ptr(signs), 1.0 / hs)
        _hip.check(_hip.lib().qp_merge_segments(args, _hip.stream_of(out)), "merge")
        torch.cuda.synchronize()
        got = to_f32(out)
        assert (np.abs(got - ref) <= 2.0 ** -7 * np.abs(ref) + 1e-5 * np.abs(ref).max(-1, keepdims=True)).all()
        assert np.abs(to_f32(lse) - want_lse).max() < 1e-4
        assert np.isnan(to_f32(wide[:, :, :off])).all() and np.isnan(to_f32(wide[:, :, hs + off:])).all()
