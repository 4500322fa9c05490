"""Batches whose longest context belongs to another sequence than the one that is split: segments and key splits are no
shorter than a floor, so the shorter sequences have fewer of them than the buffers hold, and the merge reads only those.

Tolerance: 5e-3 of fp64, as the other mixed batches of tests/test_gpu_router.py."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import i32, to_f32
from test_gpu_router import _batch, _call, _segm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int4", 64, 8, 2), ("int8", 128, 8, 2), ("int8", 256, 12, 2), ("int4", 512, 8, 2)])
def test_chunks_shorter_than_the_longest_context(device, fmt, hs, nq, nkv):
    """Chunks over 1 key to just past two split floors of 1024 keys, in one batch with a decode over 20000 keys that sets
    the host's split count."""
    import torch
    seqs = [(1, 20000), (9, 9), (12, 1023), (7, 1024), (10, 1025), (33, 2049), (2, 130)]
    views, table, q, cu, lens, qlens, ref = _batch(device, seqs, fmt, 800 + hs, nkv=nkv, hs=hs, nq=nq)
    out = torch.full_like(q, float("nan"))
    segm = _segm(device, 16, 16, nq=nq, hs=hs)
    _call(views, q, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm, 16, hs=hs)
    torch.cuda.synchronize()
    got = to_f32(out)
    for i in range(len(seqs)):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (seqs[i], O.relerr(got[sl], ref[sl]))


@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int8", 256, 24, 4), ("int4", 128, 32, 8)])
def test_decode_segments_in_a_large_mixed_batch(device, fmt, hs, nq, nkv):
    """Enough decodes of 1 to 4 tokens beside a chunk for the segment floor of 512 keys: contexts of 1 key to just past
    several floors, some sequences with one segment, one with as many as the batch's count allows."""
    import torch
    lens = [1, 31, 33, 511, 512, 513, 1024, 1025, 1537, 5000, 300, 700, 40, 64, 2048, 2049]
    seqs = [(40, 90)] + [(min(n, 1 + i % 4), n) for i, n in enumerate(lens)]
    views, table, q, cu, lens, qlens, ref = _batch(device, seqs, fmt, 820 + hs, nkv=nkv, hs=hs, nq=nq)
    out = torch.full_like(q, float("nan"))
    segm = _segm(device, 64, 16, nq=nq, hs=hs)
    _call(views, q, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm, 16, hs=hs)
    torch.cuda.synchronize()
    got = to_f32(out)
    for i in range(len(seqs)):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (seqs[i], O.relerr(got[sl], ref[sl]))


@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int4", 64, 16, 4), ("int4", 128, 16, 4), ("int8", 256, 24, 4), ("int4", 512, 16, 4)])
def test_merge_of_many_floored_segments(device, fmt, hs, nq, nkv):
    """More than 16 segments per sequence and over 1024 (row, head) pairs, with the floor of 512 keys: the merge takes the
    rows in lane groups, several batches of 8 segments for the longest contexts and one segment for the shortest."""
    import torch
    lens = [1, 31, 512, 513, 1025, 300, 64, 4095, 4096, 4097, 8200, 12000, 20000, 20001, 7, 2049]
    seqs = [(40, 90)] + [(min(n, 1 + i % 4), n) for i, n in enumerate(lens)]
    views, table, q, cu, lens, qlens, ref = _batch(device, seqs, fmt, 840 + hs, nkv=nkv, hs=hs, nq=nq)
    out = torch.full_like(q, float("nan"))
    segm = _segm(device, 68, 64, nq=nq, hs=hs)
    _call(views, q, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm, 64, hs=hs)
    torch.cuda.synchronize()
    got = to_f32(out)
    assert torch.isfinite(segm[1][:, :, 17:]).any()  # (some context has more than 16 segments)
    for i in range(len(seqs)):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (seqs[i], O.relerr(got[sl], ref[sl]))


@pytest.mark.parametrize("fmt,hs,nq,nkv", [("int4", 128, 16, 4), ("int8", 256, 24, 4)])
@pytest.mark.parametrize("T", [1, 2])
def test_library_lowers_the_segments_of_partials_in_the_workspace(device, fmt, hs, nq, nkv, T):
    """160 (sequence, KV head) pairs asking for 64 segments, with buffers for 8 of the rows: the workspace holds fewer
    segments (8 workgroups per CU in all), and the merge takes the same number. Called below the drop-in, which would
    lower the count itself."""
    import torch

    from vllm_quantpack import _hip
    from vllm_quantpack.attention import int4_kv, rht
    seqs = [(T, n) for n in [2, 33, 700, 1300] * 9 + [5000, 64, 1025, 9000]]
    views, table, q, cu, lens, qlens, ref = _batch(device, seqs, fmt, 870 + hs, nkv=nkv, hs=hs, nq=nq)
    out = torch.full_like(q, float("nan"))
    segm = _segm(device, 8, 64, nq=nq, hs=hs)
    kw = dict(cu_seqlens_q=i32(cu, device), seqused_k=i32(lens, device), block_table=i32(table, device),
              max_seqlen_q=T, max_seqlen_k=max(lens), softmax_scale=hs ** -1.5, num_segments=64,
              softmax_segm_output=segm[0], softmax_segm_max=segm[1], softmax_segm_expsum=segm[2],
              rht_signs=rht.signs(hs, device), rht_out_scale=1.0 / hs)
    need = _hip.lib().qp_attention_workspace_size(_hip.paged_cache(*views, hs), int4_kv.attention_args(q, out, **kw))
    assert 0 < need < 4 * q.shape[0] * nq * 64 * hs
    int4_kv.attend(q, *views, out, **kw)
    torch.cuda.synchronize()
    got = to_f32(out)
    assert torch.isnan(segm[0]).all()
    for i in range(len(seqs)):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (seqs[i], O.relerr(got[sl], ref[sl]))
