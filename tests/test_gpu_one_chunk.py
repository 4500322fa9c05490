"""A batch of one sequence of more than QP_DECODE_MAX_QUERY tokens goes to the prefill kernel without a route table, as the
same chunk does with one beside a decode; it asks for a workspace all the same.

Tolerance against fp64: 5e-3, as the chunks of tests/test_gpu_router.py."""
import pytest

from oracle import qp_oracle as O
from qp_testlib import i32, to_f32
from test_gpu_router import _batch, _call, _segm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,n", [(5, 5), (6, 3000), (70, 70)])
@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int4", 64, 8, 2), ("int8", 128, 8, 2), ("int8", 256, 12, 2),
                                           ("int4", 512, 8, 2), ("int8", 512, 8, 2)])
def test_single_chunk_without_a_table(device, T, n, fmt, hs, nq, nkv):
    import torch
    views, table, q, cu, lens, qlens, ref = _batch(device, [(T, n), (1, 33)], fmt, 900 + hs + T, nkv=nkv, hs=hs, nq=nq)
    segm = _segm(device, 4, 16, nq=nq, hs=hs)
    both, alone = torch.full_like(q, float("nan")), torch.full_like(q[:T], float("nan"))
    _call(views, q, both, i32(cu, device), i32(lens, device), i32(table, device), T, n, segm, 16, hs=hs)
    _call(views, q[:T], alone, i32(cu[:2], device), i32(lens[:1], device), i32(table[:1], device), T, n, segm, 16, hs=hs)
    torch.cuda.synchronize()
    assert O.relerr(to_f32(both)[:T], ref[:T]) < 5e-3
    assert O.relerr(to_f32(both)[T:], ref[T:]) < 5e-3
    assert O.relerr(to_f32(alone), ref[:T]) < 5e-3


def test_workspace_is_still_asked_for(device):
    """A plan of short sequences still refuses a longer one, also where the prefill kernel itself needs no scratch."""
    import torch

    from vllm_quantpack.attention import int4_kv
    views, table, q, cu, lens, qlens, _ = _batch(device, [(8, 8)], "int4", 930, nkv=2, hs=128, nq=8)
    segm = _segm(device, 8, 16, nq=8, hs=128)
    with pytest.raises(ValueError, match="not a batch of short sequences"):
        int4_kv.DecodePlan(q, *views, torch.empty_like(q), cu_seqlens_q=i32(cu, device), seqused_k=i32(lens, device),
                           block_table=i32(table, device), max_seqlen_q=8, softmax_scale=1.0, num_segments=16,
                           softmax_segm_output=segm[0], softmax_segm_max=segm[1], softmax_segm_expsum=segm[2])
