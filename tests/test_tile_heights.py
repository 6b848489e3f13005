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
