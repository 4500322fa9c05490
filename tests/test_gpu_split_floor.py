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
