"""What qp_prefill refuses on the host, before anything runs."""
import ctypes

import pytest


@pytest.mark.parametrize("heads,refused", [(32, False), (33, True), (64, True)])
def test_head_64_takes_at_most_32_query_heads_per_kv_head(heads, refused):
    """No query tokens, so the accepted call launches nothing."""
    from vllm_quantpack import _hip
    lib = _hip.lib()
    cache = _hip.PagedCache()
    for half, fmt in ((cache.key, 0), (cache.value, 0)):
        half.codes = half.words = 4096
        half.format = fmt
    cache.num_kv_heads, cache.head_size, cache.block_size = 1, 64, 16
    args = _hip.PrefillArgs()
    for name in ("query", "cu_seqlens_q", "seqused_k", "block_table", "out"):
        setattr(args, name, 4096)
    args.num_q_heads = heads
    st = lib.qp_prefill(ctypes.byref(cache), ctypes.byref(args), None)
    assert st == (_hip.QP_ERR_UNSUPPORTED if refused else 0), lib.qp_last_error()
    if refused:
        assert "32 query heads" in lib.qp_last_error().decode()
