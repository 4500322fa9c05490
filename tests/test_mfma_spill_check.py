"""The build checks the MFMA loops of every source that has one for spill code, whether its MFMAs are inline assembly or the
compiler's own."""
import os

import pytest

from test_boundary import _build_module


def test_sources_with_builtin_mfmas_are_checked():
    build = _build_module()
    assert build.has_mfma("s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, s, 0, 0, 0);")
    assert build.has_mfma('asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(x));')
    assert not build.has_mfma("// v_mfma in a comment")
    csrc = os.path.join(os.path.dirname(build.__file__), "csrc")
    found = [n for n in sorted(os.listdir(csrc)) if n.endswith(".hip") and build.has_mfma(open(os.path.join(csrc, n)).read())]
    assert found == ["qp_decode.hip", "qp_prefill.hip", "qp_prefill_dual.hip", "qp_prefill_i8.hip", "qp_prefill_wide.hip"]


@pytest.mark.parametrize("name,kernels", [("qp_prefill_dual", 12), ("qp_prefill_i8", 1)])
def test_built_loops_hold_no_spill_code(name, kernels):
    """The listings that the build leaves of the sources whose loops have builtin MFMAs."""
    build = _build_module()
    asm = os.path.join(build.OBJ, f"{name}.gfx.s")
    if not os.path.exists(asm):
        pytest.skip("not built")
    text = open(asm).read()
    assert build.spills_in_mfma_loops(text) == []
    assert sum(1 for hot in build.mfma_loops(text).values() if hot) >= kernels
