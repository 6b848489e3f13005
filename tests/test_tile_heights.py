"""Host side of the tile heights: what the library would launch, asked without a GPU (256 compute units then)."""
import ctypes as C
import random

import numpy as np

import therock_amd as ta
from therock_amd import _lib


def fp8(gate_only=0):
    return ta.fused_moe_traits(prec_i="fp8", prec_w="fp8", block_m=32, gate_only=gate_only)


def rows_without_routing(traits, T, E, K, H, I):
    """The tile height where the host alone decides it; 0 where the sort may choose another (the work list is then asked)."""
    t = traits.pod()
    return _lib.load().mi355_fused_moe_chosen_tile_rows(C.byref(t), T, E, K, H, I, None, None)


def test_large_tiles_do_not_come_back_as_a_second_candidate():
    """fp8 layers of so many rows per expert that even routing has the sort take the large tiles (counts rounded up to 32
    average 48) have one height, so that it is the one whose time was modelled and the down GEMM can be cut along K."""
    rng, seen = random.Random(3), 0
    while seen < 4000:
        E, K = rng.randint(4, 256), rng.randint(1, 8)
        T, H, I = int(np.exp(rng.uniform(0, 10.4))), 64 * rng.randint(8, 112), 128 * rng.randint(4, 112)
        if K > E // 2 or not 33 <= T * K / E or 3 * E * H * I > 8e9:
            continue
        seen += 1
        for gate_only in (0, 1):
            traits = fp8(gate_only)
            rows = ta.fused_moe_tile_rows(traits, T, E, K, H, I)
            assert rows_without_routing(traits, T, E, K, H, I) == rows, (T, K, E, H, I, gate_only)
    # (at few rows per expert there are two candidates)
    assert rows_without_routing(fp8(), 256, 256, 8, 7168, 2048) == 0


def test_down_gemms_that_are_cut():
    for (T, K, E, H, I), slices in (((104, 2, 5, 512, 8576), 6), ((79, 3, 7, 1088, 5376), 6), ((1481, 1, 32, 512, 3968), 4),
                                    ((1210, 4, 84, 896, 11776), 3)):
        assert ta.fused_moe_tile_rows(fp8(), T, E, K, H, I) == 320
        assert ta.fused_moe_k_slices(fp8(), T, E, K, H, I, 1 << 40) == slices


def test_down_gemms_on_the_decode_kernel():
    """Below 1.6 tiles of 256 columns a compute unit, counted over the experts that can have a row; 8-bit rows of less than 1536
    bytes below one; 16-bit weights below 8; never on the large tiles."""
    def cols(dtype, T, K, E, H, I, **kw):
        traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, prec_o="fp16" if dtype == "fp16" else "bf16", block_m=32, **kw)
        return ta.fused_moe_down_tile_cols(traits, T, E, K, H, I)
    # short rows, 1.0 to 1.6 tiles a compute unit: 8 to 14 % slower on the narrow tiles
    for case in (("int8", 65, 2, 17, 5120, 512), ("fp8", 32, 3, 17, 5184, 512), ("int8", 13, 4, 111, 1664, 576), ("fp8", 142, 6, 128, 640, 1408)):
        assert cols(*case) == 256, case
    assert cols("fp8", 97, 8, 25, 3904, 512, fused_quant=1) == 256
    # rows from 1536 bytes on; short ones below one tile; 16-bit rows
    for case in (("int8", 98, 5, 53, 1152, 1536), ("int8", 4, 5, 30, 3136, 8896), ("int8", 65, 2, 17, 2560, 512), ("bf16", 65, 2, 17, 5120, 512),
                 ("fp16", 135, 1, 203, 2304, 1216)):
        assert cols(*case) == 64, case
    # past the lines, and large tiles
    for case in (("fp8", 652, 1, 150, 704, 2048), ("int8", 64, 8, 128, 4096, 1536), ("bf16", 64, 8, 128, 4096, 1536), ("bf16", 4096, 2, 8, 4096, 14336)):
        assert cols(*case) == 256, case


def test_heights_where_the_down_gemm_runs_the_decode_kernel_past_one_tile():
    """Tiles of 128 and 320 rows stay: at 32 rows popular experts would stream their weights many times.  Of 64 rows and 32 the
    faster ones, and 32 stays where the rows are short."""
    def rows(dtype, T, K, E, H, I, **kw):
        traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, prec_o="fp16" if dtype == "fp16" else "bf16", block_m=32, **kw)
        return ta.fused_moe_tile_rows(traits, T, E, K, H, I)
    assert rows("bf16", 698, 8, 203, 576, 6848) == 128
    assert rows("bf16", 1640, 4, 243, 832, 5312, gate_only=1) == 128
    assert rows("int8", 426, 8, 124, 640, 4160, fused_quant=1) == 128
    assert rows("bf16", 1309, 1, 72, 832, 12800, weight_permute=1) == 320
    assert rows("fp16", 896, 2, 63, 1088, 10496) == 320
    assert rows("bf16", 98, 8, 35, 1856, 6912) == 32
    assert rows("fp8", 64, 5, 11, 6848, 3712) == 32
    assert rows("fp8", 132, 4, 12, 7040, 896) == 32
    assert rows("int8", 73, 5, 11, 6400, 576, gate_only=1) == 32
