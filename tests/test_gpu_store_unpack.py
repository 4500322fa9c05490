"""The store at row groups of 8 to 64 lanes (heads 64 to 512), token counts around a workgroup's, block sizes whose
division is special, and views that only allow element-wise accesses; the unpack at row and head counts of 1 and around a
workgroup's dwords. Stored bytes and unpacked values are exact."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import bf16_tensor, torch_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("hs,bs,n", [(64, 1, 33), (64, 16, 31), (128, 16, 17), (128, 48, 1), (256, 16, 9), (512, 1, 5)])
def test_store_rows_and_alignments(device, fmt, hs, bs, n):
    """The oracle's bytes; the same bytes from key and value rows at odd element offsets; and with the rotation the bytes
    of rotating first, on both."""
    import torch

    from vllm_quantpack.attention import k8v4_kv, rht
    nkv, rng = 3, np.random.default_rng(900 + hs + n)
    nb = -(-n // bs) + 2
    cell = O.int4_cell_bytes(hs) if fmt == "int4" else O.k8v4_cell_bytes(hs)
    key = O.f32_to_bf16_bits(rng.standard_normal((n, nkv, hs)).astype(np.float32) * 2)
    val = O.f32_to_bf16_bits(rng.standard_normal((n, nkv, hs)).astype(np.float32))
    slots = rng.permutation(nb * bs)[:n].astype(np.int64)
    if n > 2:
        slots[n // 2] = -1
    kt, vt = bf16_tensor(key, device), bf16_tensor(val, device)

    def odd(x):  # the same rows, each at an odd element offset of a wider one
        wide = torch.zeros((n, nkv, hs + 3), dtype=torch.bfloat16, device=device)
        wide[..., 1:1 + hs] = x
        return wide[..., 1:1 + hs]

    def stored(k, v, rotate):
        kv_np = O.new_cache(nb, nkv, bs, cell)
        t, (kc, vc, ks, vs) = torch_cache(kv_np, hs, fmt, device)
        k8v4_kv.store(None, k, v, kc, vc, torch.from_numpy(slots).to(device), k_scale_cache=ks, v_scale_cache=vs,
                      rotate=rotate)
        torch.cuda.synchronize()
        return t.cpu().numpy().view(np.uint8)

    want = O.new_cache(nb, nkv, bs, cell)
    O.store(O.int4_views(want, hs) if fmt == "int4" else O.k8v4_views(want, hs), O.bf16_bits_to_f32(key),
            O.bf16_bits_to_f32(val), slots)
    assert (stored(kt, vt, False) == want).all()
    assert (stored(odd(kt), odd(vt), False) == want).all()
    rotated = stored(rht.single_rht(kt), rht.single_rht(vt), False)
    assert (stored(kt, vt, True) == rotated).all()
    assert (stored(odd(kt), odd(vt), True) == rotated).all()


def test_store_into_byte_aligned_codes(device):
    """Code rows at odd byte addresses (a view of any layout): the codes go byte by byte, the same as aligned ones."""
    import torch

    from vllm_quantpack.attention import k8v4_kv
    n, nkv, hs, bs = 20, 2, 128, 16
    g = torch.Generator(device=device).manual_seed(5)
    k = torch.randn((n, nkv, hs), generator=g, device=device, dtype=torch.bfloat16)
    v = torch.randn((n, nkv, hs), generator=g, device=device, dtype=torch.bfloat16)
    slots = torch.arange(n, device=device) + 3
    got = []
    for shift in (0, 1):
        codes = [torch.zeros((2, bs, nkv, hs // 2 + 4 + 3 * shift), dtype=torch.uint8, device=device) for _ in range(2)]
        views = [c[..., shift:shift + hs // 2] for c in codes]
        words = [torch.zeros((2, bs, nkv), dtype=torch.float32, device=device) for _ in range(2)]
        k8v4_kv.store(None, k, v, views[0], views[1], slots, k_scale_cache=words[0], v_scale_cache=words[1])
        torch.cuda.synchronize()
        got.append([x.clone() for x in views] + words)
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("hs,nkv,bs,start,length", [(8, 1, 1, 0, 5), (8, 3, 7, 4, 1030), (64, 1, 16, 15, 129), (256, 2, 16, 1, 33)])
def test_unpack_rows(device, fmt, hs, nkv, bs, start, length):
    """bf16(fp32(code - zp) * scale) of a segment whose dwords end inside a workgroup, over blocks of any size."""
    import torch

    from vllm_quantpack.attention import int4_prefill
    g = torch.Generator(device=device).manual_seed(hs + length)
    nb = -(-(start + length) // bs) + 1
    width = hs // 2 if fmt == "int4" else hs
    codes = torch.randint(0, 256, (nb, bs, nkv, width), generator=g, device=device).to(torch.uint8)
    words = (torch.rand((nb, bs, nkv), generator=g, device=device) + 0.1).contiguous()
    row = torch.randperm(nb, generator=g, device=device).to(torch.int32)
    out = torch.full((length, nkv, hs), float("nan"), dtype=torch.bfloat16, device=device)
    view = codes if fmt == "int4" else codes.view(torch.int8)
    int4_prefill.unpack_segment(view, words, row, start, length, out)
    pos = torch.arange(start, start + length, device=device)
    blk, slot = row.long()[pos // bs], pos % bs
    c, w = codes[blk, slot], words[blk, slot]
    if fmt == "int4":
        bits = w.view(torch.int32)
        n = torch.stack((c & 15, c >> 4), -1).flatten(-2).float() - (bits & 15)[..., None].float()
        want = n * (bits & -16).view(torch.float32)[..., None]
    else:
        want = c.view(torch.int8).float() * w[..., None]
    torch.cuda.synchronize()
    assert torch.equal(out, want.to(torch.bfloat16))
