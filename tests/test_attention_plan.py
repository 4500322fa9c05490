"""How qp_attention plans a batch's split-KV partials, from the host's view of it: the workspace it asks for and what it
refuses, before anything runs."""
import ctypes

import pytest


def batch(seqs, tokens, max_q, segm_rows, nq=32, nkv=8, hs=128, segments=16):
    from vllm_quantpack import _hip
    cache = _hip.PagedCache()
    for half in (cache.key, cache.value):
        half.codes = half.words = 4096
        half.format = 0
    cache.num_kv_heads, cache.head_size, cache.block_size = nkv, hs, 16
    args = _hip.AttentionArgs()
    for name in ("query", "cu_seqlens_q", "seqused_k", "block_table", "out", "segm_output", "segm_max", "segm_expsum"):
        setattr(args, name, 4096)
    args.num_seqs, args.num_tokens, args.num_q_heads, args.max_query_len = seqs, tokens, nq, max_q
    args.max_seqlen_k, args.segm_rows, args.num_segments = 4096, segm_rows, segments
    return cache, args


def workspace(*a, **kw):
    from vllm_quantpack import _hip
    cache, args = batch(*a, **kw)
    return _hip.lib().qp_attention_workspace_size(ctypes.byref(cache), ctypes.byref(args))


@pytest.mark.parametrize("seqs,tokens,segm_rows", [(4, 32, 16), (4, 17, 16), (5, 64, 16), (1, 5, 4), (4, 64, 1)])
def test_rows_that_no_sequence_covers_are_routed(seqs, tokens, segm_rows):
    """q has more rows than the segment buffers and than 4 per sequence: the batch needs a route table (a workspace of
    at least its three arrays), as its partials cannot lie on the tokens' own rows."""
    assert workspace(seqs, tokens, 2, segm_rows) >= 3 * 256


@pytest.mark.parametrize("seqs,tokens,segm_rows", [(4, 16, 16), (4, 32, 32), (64, 64, 64), (1, 4, 4)])
def test_rows_that_fit_the_segment_buffers_need_no_workspace(seqs, tokens, segm_rows):
    assert workspace(seqs, tokens, 2, segm_rows) == 0


@pytest.mark.parametrize("change,why", [(dict(num_segments=2049), "2048 segments"), (dict(segm_output=4100), "16-byte aligned")])
def test_a_long_sequence_is_refused_for_its_segment_buffers(change, why):
    """One long sequence goes to the prefill without using the segment buffers; it is refused for them all the same, as in
    a larger batch. (The call ends there: nothing is launched on these addresses.)"""
    from vllm_quantpack import _hip
    lib = _hip.lib()
    cache, args = batch(1, 64, 64, 16)
    for name, value in change.items():
        setattr(args, name, value)
    args.workspace, args.workspace_bytes = 4096, lib.qp_attention_workspace_size(ctypes.byref(cache), ctypes.byref(args))
    st = lib.qp_attention(ctypes.byref(cache), ctypes.byref(args), None)
    assert st == _hip.QP_ERR_INVALID and why in lib.qp_last_error().decode()


@pytest.mark.parametrize("seqs,tokens,segm_rows", [(64, 64, 16), (5, 20, 19), (4, 16, 15)])
def test_rows_beyond_the_segment_buffers_are_kept_in_the_workspace(seqs, tokens, segm_rows):
    """The partials, [tokens, heads, segments, head size] and two statistics, and no route table beside them."""
    triples = tokens * 32 * 4
    assert workspace(seqs, tokens, 2, segm_rows, segments=4) == 4 * triples * 128 + 2 * 4 * triples
