"""How the head-64 / 128 prefill kernel deals a batch's row blocks to the XCDs: every block of every sequence is computed
once whatever the lengths and the number of (KV head, key split) pairs, which decides how many XCDs share a pair.

Tolerance: 5e-3 of fp64, as tests/test_gpu_router.py."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import i32, to_f32
from test_gpu_router import _batch, _call, _segm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nkv", [(8, 8), (28, 4), (6, 2), (6, 3), (6, 1)])
@pytest.mark.parametrize("hs,num_seqs", [(128, 2), (64, 7), (128, 33)])
def test_every_row_block_once(device, nq, nkv, hs, num_seqs):
    import torch
    rng = np.random.default_rng(nq + hs + num_seqs)
    # 256-row blocks: lengths on and around their edges, contexts from nothing cached to several times the longest
    edge = 256 * nkv // nq
    lens = [int(x) for x in rng.choice((5, 9, edge - 1, edge, edge + 1, 2 * edge + 3), num_seqs)]
    seqs = [(max(5, T), max(5, T) + int(rng.choice((0, 1, 40, 333)))) for T in lens]
    seqs[0] = (2 * edge + 1, 2 * edge + 1)
    if num_seqs > 2:
        seqs[1], seqs[num_seqs - 2] = (1, 700), (4, 4)                  # decodes, which the kernel skips
    views, table, q, cu, lens, qlens, ref = _batch(device, seqs, "int4", 60 + nq + hs, nkv=nkv, hs=hs, nq=nq)
    out = torch.full_like(q, float("nan"))
    segm = _segm(device, 16, 4, nq=nq, hs=hs)
    _call(views, q, out, i32(cu, device), i32(lens, device), i32(table, device), max(qlens), max(lens), segm, 4, hs=hs)
    torch.cuda.synchronize()
    got = to_f32(out)
    assert np.isfinite(got).all()
    for i in range(num_seqs):
        sl = slice(cu[i], cu[i + 1])
        assert O.relerr(got[sl], ref[sl]) < 5e-3, (i, seqs[i], O.relerr(got[sl], ref[sl]))
