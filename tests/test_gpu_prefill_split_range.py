"""Prefills over key splits whose scores lie far apart: a split whose first keys score far below its later ones keeps its
share of the merge beside a split that starts high.

Every channel of a key has the code 1 and every query channel the value 1, so a key's score in log2 units is its scale
word. Tolerance: 5e-3 of fp64, as the prefills of tests/test_gpu_parity.py."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import bf16_tensor, i32, random_cache, to_f32, torch_cache, word

pytestmark = pytest.mark.gpu


def _attend(device, fmt, hs, scores, T, G, splits, seed):
    """T query tokens of G heads over one KV head whose keys have these scores (log2 units); returns (out, fp64)."""
    import torch

    from vllm_quantpack.attention import int4_prefill
    n, bs = len(scores), 16
    kv, v = random_cache(np.random.default_rng(seed), -(-n // bs), 1, bs, hs, fmt)
    v.key[...] = 0x11 if fmt == "int4" else 1
    words = np.array([word(s, 0) if fmt == "int4" else np.float32(s).view(np.uint32) for s in scores])
    v.key_word[...] = words.reshape(v.key_word.shape)
    v.value_word[...] = (v.value_word & np.uint32(0xF)) | word(0.125, 0)
    table = np.arange(n // bs, dtype=np.int32)[None]
    _, views = torch_cache(kv, hs, fmt, device)
    scale = float(np.log(2.0)) / hs
    q = np.ones((T, G, hs), np.float32)
    qt = bf16_tensor(O.f32_to_bf16_bits(q), device)
    out = torch.full_like(qt, float("nan"))
    int4_prefill.prefill_attention(qt, *views, out, cu_seqlens_q=i32([0, T], device), seqused_k=i32([n], device),
                                   block_table=i32(table, device), max_seqlen_q=T, softmax_scale=scale,
                                   num_splits=splits)
    torch.cuda.synchronize()
    K, V = O.dequant_f64(v, table[0], n)
    return to_f32(out), O.attention_f64(q, K, V, n, scale)


@pytest.mark.parametrize("fmt,hs,G", [("int4", 64, 4), ("int8", 64, 4), ("int4", 128, 4), ("int8", 128, 4),
                                      ("int4", 128, 8), ("int4", 256, 6), ("int4", 512, 4), ("int8", 512, 4)])
@pytest.mark.parametrize("order", [1, -1], ids=["rising-first", "rising-last"])
def test_splits_whose_maxima_rise_after_their_first_keys(device, fmt, hs, G, order):
    """1024 keys that start at 1 and go on at 119, and 1024 that hold one key at 128: the 992 keys at 119 weigh twice as
    much as the one at 128, though each is 2^9 below it. In the middle a split without anything near them."""
    rising = np.concatenate((np.full(32, 1.0), np.full(992, 119.0)))
    high = np.concatenate(([128.0], np.full(1023, 1.0)))
    scores = np.concatenate([(rising, np.full(1024, 2.0), high)[::order][i] for i in range(3)])
    out, ref = _attend(device, fmt, hs, scores, 7, G, 3, 40 + hs)
    assert np.isfinite(out).all()
    assert O.relerr(out, ref) < 5e-3, O.relerr(out, ref)


@pytest.mark.parametrize("fmt,hs,G", [("int4", 64, 4), ("int8", 64, 4), ("int4", 128, 4), ("int8", 128, 8), ("int4", 512, 4)])
def test_splits_that_run_again_beside_others(device, fmt, hs, G):
    """Two splits whose later keys score 250 to 300 above their first (past the headroom, so their workgroups start again
    with the true maxima) and one that is high from its first key on and does not."""
    a = np.concatenate((np.full(100, 1.0), [300.0], np.full(923, 2.0)))
    b = np.concatenate((np.full(32, 3.0), np.full(492, 251.0), np.full(500, 291.0)))
    c = np.concatenate((np.full(40, 292.0), np.full(984, 280.0)))
    out, ref = _attend(device, fmt, hs, np.concatenate((a, b, c)), 5, G, 3, 60 + hs)
    assert np.isfinite(out).all()
    assert O.relerr(out, ref) < 5e-3, O.relerr(out, ref)
