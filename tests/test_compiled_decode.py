"""What the compiler made of the decode GEMM.  A workgroup lives some 10 us there, so that setting up scratch memory shows."""
import pytest

from tests import compiled_kernels as ck

pytestmark = pytest.mark.skipif(not ck.tools_there(), reason="ROCm's LLVM tools are not installed")


def test_no_form_uses_scratch_memory():
    said = {name: notes for name, notes in ck.kernels().items() if "moe_gemm_decode_kernel" in name}
    # gate+up and down of bf16, fp16, fp8 and int8, and bf16 by int8; two token blocks where there are (not fp8, nor bf16 by
    # int8); two weight layouts
    assert len(said) == 30
    spilled = {name: notes for name, notes in said.items() if notes["private_segment_fixed_size"] or notes["vgpr_spill_count"]}
    assert not spilled, spilled
