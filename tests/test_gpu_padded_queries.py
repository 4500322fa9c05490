"""Batches of short sequences whose q has more rows than the sequences cover (a padded batch), with segment buffers that
hold every row, the sequences' rows only, or fewer.

Tolerance: 5e-3 of fp64, as tests/test_gpu_router.py."""
import pytest

from oracle import qp_oracle as O
from qp_testlib import i32, to_f32
from test_gpu_router import _batch, _call, _segm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int4", 64, 8, 2), ("int4", 128, 8, 2), ("int8", 256, 12, 2), ("int4", 512, 8, 2)])
@pytest.mark.parametrize("seqs,rows,buffers", [(4, 32, 16), (5, 64, 16), (5, 64, 3), (4, 32, 32), (1, 9, 1)])
def test_rows_past_the_sequences(device, seqs, rows, buffers, fmt, hs, nq, nkv):
    import torch
    shapes = [(2, 700), (1, 1), (2, 1300), (1, 33), (2, 64)][:seqs]
    views, table, q, cu, lens, qlens, ref = _batch(device, shapes, fmt, 610 + hs, nkv=nkv, hs=hs, nq=nq)
    covered = q.shape[0]
    padded = torch.full((rows, nq, hs), 7.0, dtype=torch.bfloat16, device=device)
    padded[:covered] = q
    out = torch.full_like(padded, float("nan"))
    segm = _segm(device, buffers, 16, nq=nq, hs=hs)
    for x in segm:
        x.zero_()  # (rows that no sequence covers have partials from nowhere: their output is not looked at)
    _call(views, padded, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm, 16,
          hs=hs)
    torch.cuda.synchronize()
    got = to_f32(out)[:covered]
    for i in range(seqs):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (i, O.relerr(got[sl], ref[sl]))


@pytest.mark.parametrize("segments", [16, 64])  # (a merge of few segments, and of many)
@pytest.mark.parametrize("rows,buffers", [(9, 3), (20, 8), (33, 3)])
def test_output_of_rows_past_the_sequences(device, rows, buffers, segments):
    """Where the partials go to the workspace, rows of q that no sequence covers have none: their output is left alone."""
    import torch
    shapes = [(2, 700), (1, 1), (2, 1300), (1, 33), (2, 64)]
    views, table, q, cu, lens, qlens, ref = _batch(device, shapes, "int4", 650, nkv=2, hs=128, nq=8)
    covered = q.shape[0]
    padded = torch.ones((rows, 8, 128), dtype=torch.bfloat16, device=device)
    padded[:covered] = q
    out = torch.full_like(padded, -3.0)
    segm = _segm(device, buffers, segments, nq=8, hs=128)
    _call(views, padded, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm,
          segments, hs=128)
    torch.cuda.synchronize()
    assert O.relerr(to_f32(out)[:covered], ref) < 5e-3
    assert (out[covered:] == -3.0).all()


def test_plan_refuses_rows_past_the_buffers(device):
    """A prepared decode step on the tokens' own rows needs a buffer row for each: refused when it is made."""
    import torch

    from vllm_quantpack.attention import int4_kv
    views, table, q, cu, lens, qlens, _ = _batch(device, [(1, 40)] * 4, "int4", 640, nkv=2, hs=128, nq=8)
    padded = torch.cat((q, q, q, q, q, q, q, q))
    segm = _segm(device, 16, 16, nq=8, hs=128)
    with pytest.raises(ValueError, match="fit the segment buffers"):
        int4_kv.DecodePlan(padded, *views, torch.empty_like(padded), cu_seqlens_q=i32(cu, device),
                           seqused_k=i32(lens, device), block_table=i32(table, device), max_seqlen_q=1,
                           softmax_scale=1.0, num_segments=16, softmax_segm_output=segm[0], softmax_segm_max=segm[1],
                           softmax_segm_expsum=segm[2])
