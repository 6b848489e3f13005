"""What the compiler made of the decode and the small-tile GEMMs: scratch memory, which a decode workgroup of some 10 us notices, and
the registers that decide how many workgroups a compute unit runs."""
import re

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


def test_small_tiles_leave_room_for_their_workgroups():
    """Four workgroups of four waves a compute unit in tiles of 32 rows (128 registers), three in tiles of 64 (168; the fp8 down
    GEMM, whose rows bring block scales, two)."""
    seen = 0
    for name, notes in ck.kernels().items():
        m = re.search(r"15moe_gemm_kernelILi(\d)ELb(\d)ELi([12])E", name)
        if not m:
            continue
        mode, gemm0, blocks = (int(x) for x in m.groups())
        most = 128 if blocks == 1 else 256 if (mode, gemm0) == (1, 0) else 168
        assert notes["vgpr_count"] <= most and notes["private_segment_fixed_size"] == 0, (name, notes)
        seen += 1
    assert seen == 18
