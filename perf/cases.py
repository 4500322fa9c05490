"""The calls whose time matters to a program that serves a model over an int4 or k8v4 KV cache, as measurable cases.

A serving engine makes three kinds of calls per layer: it stores the new tokens' keys and values in the paged cache
(`reshape_and_cache_int4`), it attends over the cache (`unified_attention_int4`: decode steps, prompt chunks, batches
of prompts and batches that mix them), and, where other code wants bf16 keys and values, it unpacks a cache segment
(`unpack_segment`). `listed()` holds the ordinary sizes of these, `draw()` gives others of the same ranges, `prepare()`
makes what the engine has in hand before the call and `run()` is the call.

An attention case is a batch of `decodes` sequences of up to `decode_tokens` query tokens (1 plus the drafts that are
verified with it) over up to `decode_context` cached tokens, followed by `chunks` sequences of up to `chunk_tokens`
query tokens that extend `chunk_cached` cached tokens; with `ragged` the lengths differ, drawn from the number `lens`.
`rows` is the number of rows of the split-KV segment buffers the engine allocated once: 0 for one per query token, or
128 / KV heads, the size an engine that allocates for its smallest batches has.
"""
import math
import random
import sys

import torch

sys.path.insert(0, "vllm-quantpack_amd")

from vllm_quantpack.attention import int4_kv, int4_prefill, k8v4_kv  # noqa: E402

DEVICE = "cuda"


def attention(name, key, nq, nkv, hs, bs=16, decodes=0, decode_tokens=1, decode_context=0, chunks=0, chunk_tokens=0,
              chunk_cached=0, ragged=False, lens=0, rows=0):
    return dict(name=name, op="attention", key=key, nq=nq, nkv=nkv, hs=hs, bs=bs, decodes=decodes,
                decode_tokens=decode_tokens, decode_context=decode_context, chunks=chunks, chunk_tokens=chunk_tokens,
                chunk_cached=chunk_cached, ragged=ragged, lens=lens, rows=rows)


def listed():
    return [
        # one user, a short conversation, one token at a time: the smallest decode step, set by latency
        attention("decode-4k", "int4", 24, 4, 256, decodes=1, decode_tokens=1, decode_context=4096, rows=32),
        # one user over a long document, one draft token verified per step
        attention("decode-128k-t2", "int4", 24, 4, 256, decodes=1, decode_tokens=2, decode_context=131072, rows=32),
        # the same over a very long context with three drafts: more query rows per KV head than one 16-row tile
        attention("decode-256k-t4", "int4", 24, 4, 256, decodes=1, decode_tokens=4, decode_context=262144, rows=32),
        # a batch of requests of different ages on the k8v4 cache, some with a draft token
        attention("decode-b32-k8v4", "int8", 24, 4, 256, decodes=32, decode_tokens=2, decode_context=65536,
                  ragged=True, lens=4),
        # many chat requests of different ages at head 128, one token each, on an engine whose segment buffers hold
        # fewer rows than the batch has tokens
        attention("decode-b64-h128", "int4", 32, 8, 128, decodes=64, decode_tokens=1, decode_context=8192, ragged=True,
                  lens=5, rows=16),
        # one chunk of a long prompt, most of it cached: the largest call
        attention("chunk-128k", "int4", 24, 4, 256, chunks=1, chunk_tokens=1024, chunk_cached=131072, rows=32),
        # a chunk of a prompt of ordinary length at head 128 with 8 query heads per KV head, in 32-token blocks
        attention("chunk-16k-h128", "int4", 64, 8, 128, bs=32, chunks=1, chunk_tokens=2048, chunk_cached=16384, rows=16),
        # new prompts of different lengths in one batch, nothing cached
        attention("prompts-h128", "int4", 32, 8, 128, chunks=8, chunk_tokens=2048, ragged=True, lens=8, rows=16),
        # continuous batching: decoding requests beside a chunk of a new prompt, on the k8v4 cache
        attention("mixed-k8v4", "int8", 24, 4, 256, decodes=24, decode_tokens=1, decode_context=16384, chunks=1,
                  chunk_tokens=509, chunk_cached=2048, ragged=True, lens=9, rows=32),
        # a prompt of a small model: head 64
        attention("chunk-4k-h64", "int8", 32, 8, 64, chunks=1, chunk_tokens=512, chunk_cached=4096, rows=16),
        # the new tokens of a prompt batch written to the cache
        dict(name="store-4k-h128", op="store", key="int4", nq=32, nkv=8, hs=128, bs=16, tokens=4096),
        # a 16384-token segment of keys and values unpacked to bf16
        dict(name="unpack-16k", op="unpack", key="int4", nkv=4, hs=256, bs=16, start=16384, length=16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


HEADS = {64: ((32, 8),), 128: ((32, 8), (64, 8), (28, 4)), 256: ((24, 4), (32, 2), (16, 4)), 512: ((16, 2),)}


def draw(rng):
    """A case of the same ranges. Its work is held below the largest listed case's."""
    hs = rng.choice((64, 128, 128, 256, 256, 256, 512))
    nq, nkv = rng.choice(HEADS[hs])
    key = rng.choice(("int4", "int4", "int8"))
    bs = rng.choice((16, 16, 16, 32, 48))
    kind = rng.choice(("decode", "decode", "batch", "batch", "chunk", "chunk", "prompts", "mixed", "store", "unpack"))
    if kind == "store":
        case = dict(op="store", key=key, nq=nq, nkv=nkv, hs=hs, bs=bs, tokens=_log_int(rng, 1, 8192))
        return case
    if kind == "unpack":
        length = _log_int(rng, 1000, 16384)
        return dict(op="unpack", key=key, nkv=nkv, hs=hs, bs=bs, start=rng.randrange(0, 16384), length=length)
    c = dict(op="attention", key=key, nq=nq, nkv=nkv, hs=hs, bs=bs, decodes=0, decode_tokens=1, decode_context=0,
             chunks=0, chunk_tokens=0, chunk_cached=0, ragged=kind != "decode", lens=rng.randrange(10 ** 6),
             rows=128 // nkv)
    if kind == "decode":
        c.update(decodes=1, decode_tokens=rng.randint(1, 4), decode_context=_log_int(rng, 256, 262144))
    elif kind == "batch":
        c.update(decodes=_log_int(rng, 2, 128), decode_tokens=rng.choice((1, 1, 2)),
                 decode_context=_log_int(rng, 1024, 65536), rows=rng.choice((0, 128 // nkv)))
    elif kind == "chunk":
        c.update(chunks=1, chunk_tokens=_log_int(rng, 33, 2048), chunk_cached=_log_int(rng, 256, 131072))
    elif kind == "prompts":
        c.update(chunks=rng.randint(1, 12), chunk_tokens=_log_int(rng, 128, 2048))
    else:
        c.update(decodes=_log_int(rng, 2, 64), decode_tokens=rng.choice((1, 1, 2)),
                 decode_context=_log_int(rng, 1024, 32768), chunks=rng.choice((1, 1, 2)),
                 chunk_tokens=_log_int(rng, 33, 1024), chunk_cached=_log_int(rng, 16, 8192))
    if c["chunks"] == 0:
        c["bs"] = 16 if c["decodes"] == 1 else bs
    # the largest listed chunk has 3.3 TFLOP; heads 64 and 512 are drawn smaller, in keeping with the models that have
    # them
    limit = 1.5e12 if hs in (128, 256) else 1e11
    while work(c)["flops"] > limit:
        for part in ("chunk_cached", "chunk_tokens", "decode_context"):
            c[part] -= c[part] // 4
    while work(c)["bytes"] > 8e8:
        c["decode_context"] -= c["decode_context"] // 4
    return c


# ------------------------------------------------------------------------------------------- shapes of a case

def lengths(case):
    """(query tokens, context including them) of every sequence of an attention case, decoding ones first."""
    rng = random.Random(case["lens"])
    seqs = []
    for _ in range(case["decodes"]):
        t, n = case["decode_tokens"], case["decode_context"]
        if case["ragged"]:
            t, n = rng.randint(1, t), _log_int(rng, max(8, n // 32), n)
        seqs.append((t, max(t, n)))
    for _ in range(case["chunks"]):
        t = case["chunk_tokens"]
        if case["ragged"] and case["chunks"] > 1:
            t = max(5, _log_int(rng, max(5, t // 16), t))
        seqs.append((t, t + case["chunk_cached"]))
    return seqs


def _cell(case):
    return (case["hs"] // 2 if case["key"] == "int4" else case["hs"]) + case["hs"] // 2 + 8


def work(case):
    if case["op"] == "store":
        rows = case["tokens"] * case["nkv"]
        return {"bytes": rows * (2 * 2 * case["hs"] + _cell(case)) + 8 * case["tokens"],
                "flops": 2 * rows * case["hs"] * math.log2(case["hs"])}
    if case["op"] == "unpack":
        rows = case["length"] * case["nkv"]
        return {"bytes": rows * (_cell(case) + 2 * 2 * case["hs"]), "flops": 2 * 2 * rows * case["hs"]}
    cells = pairs = rows = blocks = 0
    for t, n in lengths(case):
        cells += n * case["nkv"]
        blocks += -(-n // case["bs"])
        rows += t * case["nq"]
        pairs += (t * (n - t) + t * (t + 1) // 2) * case["nq"]
    return {"bytes": cells * _cell(case) + 4 * blocks + 2 * rows * 2 * case["hs"], "flops": 4 * case["hs"] * pairs}


# ------------------------------------------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _fill_cache(case, blocks, gen):
    """A byte cache (blocks, KV heads, block size, cell) as the store leaves it for normal keys and values: codes of
    rotated rows (normal, their largest of hs channels at the end of the code range), one scale word per token and
    head."""
    hs, half = case["hs"], case["hs"] // 2
    shape = (blocks, case["nkv"], case["bs"])
    kv = torch.empty((*shape, _cell(case)), dtype=torch.uint8, device=DEVICE)

    def normal(*size):
        return torch.randn(size, generator=gen, device=DEVICE)

    def sigma():                      # of a rotated row: the rotation is unnormalised
        return math.sqrt(hs) * torch.exp(0.25 * normal(*shape))

    def int4(at):
        zp = torch.round(7.5 + 0.7 * normal(*shape)).clamp_(0, 15)
        u = torch.round(normal(*shape, hs).mul_(2.7).add_(zp[..., None])).clamp_(0, 15).to(torch.uint8)
        kv[..., at:at + half] = u[..., 0::2] | (u[..., 1::2] << 4)
        word = ((sigma() / 2.7).view(torch.int32) & -16) | zp.to(torch.int32)
        kv[..., at + half:at + half + 4] = word[..., None].view(torch.uint8)

    if case["key"] == "int4":
        int4(0)
        int4(half + 4)
    else:
        code = torch.round(normal(*shape, hs).mul_(45.0)).clamp_(-127, 127).to(torch.int8)
        kv[..., :hs] = code.view(torch.uint8)
        kv[..., hs:hs + 4] = (sigma() / 45.0)[..., None].view(torch.uint8)
        int4(hs + 4)
    return kv


def _views(case, kv):
    return k8v4_kv.views(kv, case["hs"]) if case["key"] == "int8" else k8v4_kv.int4_views(kv, case["hs"])


def _bf16(gen, *size):
    return torch.randn(size, generator=gen, device=DEVICE).to(torch.bfloat16)


def _blocks(case):
    """Cache blocks of a case."""
    if case["op"] == "store":
        return -(-case["tokens"] // case["bs"]) + 64
    if case["op"] == "unpack":
        return -(-(case["start"] + case["length"]) // case["bs"])
    return sum(-(-n // case["bs"]) for _, n in lengths(case))


def _inputs(case, seed):
    """(cache, other inputs) of a case, from the seed alone."""
    gen = _generator(seed)
    blocks = _blocks(case)
    kv = _fill_cache(case, blocks, gen)
    order = torch.randperm(blocks, generator=gen, device=DEVICE)
    if case["op"] == "store":
        # keys and values as slices of the fused projection's output, slots in the blocks the engine handed out
        qkv = _bf16(gen, case["tokens"], case["nq"] + 2 * case["nkv"], case["hs"])
        pos = torch.arange(case["tokens"], device=DEVICE)
        slots = order[pos // case["bs"]] * case["bs"] + pos % case["bs"]
        return kv, dict(key=qkv[:, case["nq"]:case["nq"] + case["nkv"]], value=qkv[:, case["nq"] + case["nkv"]:],
                        slots=slots)
    order = order.to(torch.int32)
    if case["op"] == "unpack":
        return kv, dict(row=order)
    seqs = lengths(case)
    table = torch.zeros((len(seqs), max(-(-n // case["bs"]) for _, n in seqs)), dtype=torch.int32, device=DEVICE)
    at = 0
    for i, (_, n) in enumerate(seqs):
        nb = -(-n // case["bs"])
        table[i, :nb] = order[at:at + nb]
        at += nb
    q = _bf16(gen, sum(t for t, _ in seqs), case["nq"], case["hs"])
    return kv, dict(q=q, table=table)


def prepare(case, seed):
    kv, x = _inputs(case, seed)
    state = dict(case=case, kv=kv, views=_views(case, kv), **x)
    if case["op"] == "unpack":
        shape = (case["length"], case["nkv"], case["hs"])
        state["out"] = [torch.empty(shape, dtype=torch.bfloat16, device=DEVICE) for _ in range(2)]
    if case["op"] == "attention":
        seqs = lengths(case)
        starts = [0]
        for t, _ in seqs:
            starts.append(starts[-1] + t)
        segments = int4_kv.segments_for(torch.cuda.get_device_properties(0).multi_processor_count)
        rows = case["rows"] or starts[-1]
        state.update(
            out=torch.empty_like(x["q"]), segments=segments,
            cu=torch.tensor(starts, dtype=torch.int32, device=DEVICE),
            used=torch.tensor([n for _, n in seqs], dtype=torch.int32, device=DEVICE),
            max_q=max(t for t, _ in seqs), max_k=max(n for _, n in seqs),
            segm_output=torch.empty((rows, case["nq"], segments, case["hs"]), dtype=torch.float32, device=DEVICE),
            segm_max=torch.empty((rows, case["nq"], segments), dtype=torch.float32, device=DEVICE),
            segm_sum=torch.empty((rows, case["nq"], segments), dtype=torch.float32, device=DEVICE))
    return state


def run(state):
    case = state["case"]
    kc, vc, ks, vs = state["views"]
    if case["op"] == "store":
        int4_kv.reshape_and_cache_int4(state["key"], state["value"], kc, vc, state["slots"], k_scale_cache=ks,
                                       v_scale_cache=vs)
        return state["kv"]
    if case["op"] == "unpack":
        for codes, words, out in ((kc, ks, state["out"][0]), (vc, vs, state["out"][1])):
            int4_prefill.unpack_segment(codes, words, state["row"], case["start"], case["length"], out)
        return state["out"]
    int4_kv.unified_attention_int4(
        state["q"], kc, vc, state["out"], cu_seqlens_q=state["cu"], max_seqlen_q=state["max_q"],
        seqused_k=state["used"], max_seqlen_k=state["max_k"], softmax_scale=case["hs"] ** -0.5, window_size=(-1, -1),
        block_table=state["table"], softcap=0.0, sinks=None, alibi_slopes=None, use_alibi_sqrt=False, qq_bias=None,
        output_scale=None, mm_prefix_range=None, k_scale_cache=ks, v_scale_cache=vs, seq_threshold_3D=case["rows"],
        num_par_softmax_segments=state["segments"], softmax_segm_output=state["segm_output"],
        softmax_segm_max=state["segm_max"], softmax_segm_expsum=state["segm_sum"])
    return state["out"]


# ------------------------------------------------------------------------------------- 64-bit results, tolerances

def tolerance(case):
    if case["op"] != "attention":
        return "exact"               # stored bytes and exactly rounded products
    # bf16 queries after the rotation, bf16 probabilities, one bf16 rounding of the output
    return {"rel": 1e-2}


def _signs(hs):
    """The rotation's +/-1 diagonal: bit 0 of an integer hash of the channel."""
    out = []
    for x in range(hs):
        x ^= x >> 16
        x = x * 0x7FEB352D & 0xFFFFFFFF
        x ^= x >> 15
        x = x * 0x846CA68B & 0xFFFFFFFF
        x ^= x >> 16
        out.append(-1.0 if x & 1 else 1.0)
    return torch.tensor(out, dtype=torch.float64, device=DEVICE)


def _hadamard(hs):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEVICE)
    while h.shape[0] < hs:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _dequant(case, cells, value):
    """Rows of cells (..., cell) to float64 channels of their key or value half."""
    hs, half = case["hs"], case["hs"] // 2
    kbytes = half if case["key"] == "int4" else hs
    at = kbytes + 4 if value else 0
    if not value and case["key"] == "int8":
        scale = cells[..., hs:hs + 4].contiguous().view(torch.float32).to(torch.float64)
        return cells[..., :hs].view(torch.int8).to(torch.float64) * scale
    word = cells[..., at + half:at + half + 4].contiguous().view(torch.int32)
    scale = (word & -16).view(torch.float32).to(torch.float64)
    b = cells[..., at:at + half]
    u = torch.stack((b & 15, b >> 4), -1).flatten(-2).to(torch.float64)
    return (u - (word & 15).to(torch.float64)) * scale


def exact(case, seed):
    if case["op"] == "store":
        return None
    kv, x = _inputs(case, seed)
    hs, nkv, bs = case["hs"], case["nkv"], case["bs"]
    if case["op"] == "unpack":
        pos = torch.arange(case["start"], case["start"] + case["length"], device=DEVICE)
        cells = kv[x["row"].long()[pos // bs], :, pos % bs]
        return [_dequant(case, cells, value) for value in (False, True)]
    signs, had = _signs(hs), _hadamard(hs)
    group = case["nq"] // nkv
    out = torch.zeros(x["q"].shape, dtype=torch.float64, device=DEVICE)
    q0 = 0
    for i, (t, n) in enumerate(lengths(case)):
        pos = torch.arange(n, device=DEVICE)
        block, slot = x["table"][i].long()[pos // bs], pos % bs
        limit = torch.arange(n - t, n, device=DEVICE).repeat_interleave(group)
        for h in range(nkv):
            cells = kv[block, h, slot]
            k, v = _dequant(case, cells, False), _dequant(case, cells, True)
            q = x["q"][q0:q0 + t, h * group:(h + 1) * group].to(torch.float64)
            rows = ((q * signs) @ had).reshape(t * group, hs)
            res = torch.empty_like(rows)
            for r in range(0, rows.shape[0], 1024):
                s = rows[r:r + 1024] @ k.T * (hs ** -0.5 / hs)
                s.masked_fill_(pos[None, :] > limit[r:r + 1024, None], -math.inf)
                res[r:r + 1024] = torch.softmax(s, -1) @ v
            out[q0:q0 + t, h * group:(h + 1) * group] = ((res @ had) * signs / hs).reshape(t, group, hs)
        q0 += t
    return out
