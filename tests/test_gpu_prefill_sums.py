"""The softmax of the prefill kernel at heads 64 and 128 beyond its outputs on ordinary inputs: the row sums its split
partials hold, and the scales at which a score or a value carries nothing. (SHAPES: those whose sums are of unrounded
probabilities; at head 128 below 8 query heads per KV head they are of the rounded ones.)

Tolerances: a row's log-sum-exp in log2 units within 1e-4 of fp64 (fp32 scores of up to 64 units: 2^-18 for the rounding of
their reference and as much for each of the score's two products); outputs within 5e-3 of fp64, as the prefills of
tests/test_gpu_parity.py."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import bf16_tensor, i32, random_cache, to_f32, torch_cache

pytestmark = pytest.mark.gpu

SHAPES = [("int4", 64, 4, 2), ("int8", 64, 8, 2), ("int4", 128, 16, 2), ("int8", 128, 16, 2)]


def _case(device, fmt, hs, nq, nkv, n, T, scale, seed, change=None):
    """(q, views, host views, keyword arguments of the call) of T query tokens over n keys; change(host views) edits the
    cache first."""
    rng = np.random.default_rng(seed)
    kv, v = random_cache(rng, -(-n // 16), nkv, 16, hs, fmt)
    if change:
        change(v)
    _, views = torch_cache(kv, hs, fmt, device)
    q = O.f32_to_bf16_bits(rng.standard_normal((T, nq, hs)).astype(np.float32))
    table = np.arange(-(-n // 16), dtype=np.int32)[None]
    kw = dict(cu_seqlens_q=i32([0, T], device), seqused_k=i32([n], device), block_table=i32(table, device),
              max_seqlen_q=T, softmax_scale=scale)
    return q, views, v, table[0], kw


@pytest.mark.parametrize("fmt,hs,nq,nkv", SHAPES)
@pytest.mark.parametrize("n", [12, 300])
def test_row_sums_are_those_of_unrounded_probabilities(device, fmt, hs, nq, nkv, n):
    """m + log2(l) of every row, over few keys (where a rounding of the probabilities to bf16, 2^-9 each, would show) and
    over several tiles."""
    import torch

    from vllm_quantpack import _hip
    from vllm_quantpack.attention import int4_prefill
    T, splits, scale = 12, 2, hs ** -0.5
    q, views, v, row, kw = _case(device, fmt, hs, nq, nkv, n, T, scale, 840 + hs + n)
    qt = bf16_tensor(q, device)
    out = torch.empty_like(qt)
    cache, args = int4_prefill._prefill_args(qt, *views, out, kw["cu_seqlens_q"], kw["seqused_k"], kw["block_table"], T,
                                             scale, n, splits)
    rows = T * nq * splits
    ws = torch.full((rows * (hs + 2),), float("nan"), dtype=torch.float32, device=device)
    assert _hip.lib().qp_prefill_workspace_size(cache, args) == 4 * ws.numel()
    args.workspace, args.workspace_bytes = ws.data_ptr(), 4 * ws.numel()
    _hip.check(_hip.lib().qp_prefill(cache, args, _hip.stream_of(qt)), "prefill")
    torch.cuda.synchronize()
    stats = ws[rows * hs:].cpu().numpy().astype(np.float64).reshape(2, T, nq, splits)
    K, _ = O.dequant_f64(v, row, n)
    seg = O.segment_length(n, splits, 32)
    for s in range(splits):
        for t in range(T):
            last = min((s + 1) * seg, n - T + t + 1)
            if s * seg >= n or last <= s * seg:
                continue
            keys = np.repeat(K[s * seg:last], nq // nkv, axis=1)
            score = np.einsum("hc,khc->hk", O.bf16_bits_to_f32(q[t]).astype(np.float64), keys) * scale * np.log2(np.e)
            got = stats[0, t, :, s] + np.log2(stats[1, t, :, s])
            assert np.abs(got - np.log2(np.exp2(score).sum(axis=1))).max() < 1e-4, (t, s)


@pytest.mark.parametrize("fmt,hs,nq,nkv", SHAPES + [("int4", 128, 4, 1), ("int8", 128, 4, 1)])
@pytest.mark.parametrize("scale", [0.0, -0.05, 1e-32])
def test_scales_without_a_sign_or_a_size(device, fmt, hs, nq, nkv, scale):
    """A softmax scale of 0 (all keys alike), below 0, and so small that no score differs."""
    import torch

    from vllm_quantpack.attention import int4_prefill
    T, n = 9, 150
    q, views, v, row, kw = _case(device, fmt, hs, nq, nkv, n, T, scale, 860 + hs)
    out = torch.full((T, nq, hs), float("nan"), dtype=torch.bfloat16, device=device)
    int4_prefill.prefill_attention(bf16_tensor(q, device), *views, out, **kw)
    torch.cuda.synchronize()
    K, V = O.dequant_f64(v, row, n)
    ref = O.attention_f64(O.bf16_bits_to_f32(q), K, V, n, scale)
    assert O.relerr(to_f32(out), ref) < 5e-3, O.relerr(to_f32(out), ref)


@pytest.mark.parametrize("fmt,hs,nq,nkv", SHAPES)
def test_keys_whose_value_scale_is_zero(device, fmt, hs, nq, nkv):
    """A key with a value scale of 0 takes its share of the softmax and adds nothing to the output."""
    import torch

    from vllm_quantpack.attention import int4_prefill
    T, n, scale = 9, 150, hs ** -0.5

    def change(v):
        v.value_word[:, ::3] = 0

    q, views, v, row, kw = _case(device, fmt, hs, nq, nkv, n, T, scale, 880 + hs, change)
    out = torch.full((T, nq, hs), float("nan"), dtype=torch.bfloat16, device=device)
    int4_prefill.prefill_attention(bf16_tensor(q, device), *views, out, **kw)
    torch.cuda.synchronize()
    K, V = O.dequant_f64(v, row, n)
    ref = O.attention_f64(O.bf16_bits_to_f32(q), K, V, n, scale)
    assert O.relerr(to_f32(out), ref) < 5e-3, O.relerr(to_f32(out), ref)
