"""The prefill kernel with two waves per SIMD (heads 64 and 128, csrc/qp_prefill_dual.hip) at the sizes where its tiling
can go wrong: contexts around its 32-key sub-tiles and 64-key tiles, chunks that end around a wave's 32 and a
workgroup's 256 (token, query head) rows, key splits that end mid-tile, and scores that force its second pass.

Tolerances: the ones tests/test_gpu_parity.py derives for prefills (5e-3 of fp64: bf16 probabilities and output; 1e-2 of
the emulated reference kernel, per row)."""
import numpy as np
import pytest

from oracle import qp_oracle as O
from qp_testlib import assert_emulation
from test_gpu_parity import _prefill_case

pytestmark = pytest.mark.gpu


def _check(out, emu, ref, lens):
    assert np.isfinite(out).all()
    at = 0
    for T, n in lens:
        sl = slice(at, at + T)
        assert_emulation(out[sl], emu[sl], (T, n))
        assert O.relerr(out[sl], ref[sl]) < 5e-3, (T, n, O.relerr(out[sl], ref[sl]))
        at += T


@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("hs", [64, 128])
@pytest.mark.parametrize("layout,bs,splits", [("hnd", 16, 1), ("hnd", 48, 3), ("nhd", 16, 2)])
def test_context_lengths_around_the_tiles(device, fmt, hs, layout, bs, splits):
    """7 query tokens over contexts of 1 to 4 tiles, each one key short of, at and past a sub-tile's or tile's end (the
    chunk's own keys, masked, are in the last one or two sub-tiles), one split or splits of whole 32-key sub-tiles."""
    rng = np.random.default_rng(700 + hs + bs + (fmt == "int8"))
    lens = [(7, n) for n in (7, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 129, 191, 193, 255, 257)]
    _check(*_prefill_case(device, rng, fmt, lens, layout=layout, bs=bs, nq=16, nkv=2, hs=hs, splits=splits), lens)


@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("hs,nq,nkv", [(64, 8, 2), (128, 8, 2), (128, 14, 2)])
def test_rows_around_a_wave_and_a_workgroup(device, fmt, hs, nq, nkv):
    """Chunks of 4 or 7 rows per token that end just before, at and after 32, 64 and 256 rows (waves without rows only
    copy and unpack), in one batch, with nothing cached and over cached keys."""
    rng = np.random.default_rng(720 + hs + nq + (fmt == "int8"))
    lens = [(5, 40), (8, 8), (9, 100), (16, 70), (17, 17), (63, 300), (64, 64), (65, 200), (73, 73), (129, 140)]
    _check(*_prefill_case(device, rng, fmt, lens, nq=nq, nkv=nkv, hs=hs), lens)


@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("hs", [64, 128])
def test_scores_that_force_the_second_pass(device, fmt, hs):
    """Keys with scales 2^7 to 2^12 far into the context raise scores past the first sub-tile's maximum by more than the
    kernel's bias and headroom together: the workgroup runs its split again with the true maxima."""
    rng = np.random.default_rng(740 + hs)
    lens = [(40, 900), (9, 700)]
    out, emu, ref = _prefill_case(device, rng, fmt, lens, nq=8, nkv=2, hs=hs, splits=1,
                                  big_keys=[(300, 2.0 ** 7), (421, 2.0 ** 12)])
    assert np.isfinite(out).all()
    assert O.relerr(out, ref) < 5e-3, O.relerr(out, ref)
