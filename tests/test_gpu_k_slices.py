"""The down GEMM cut along K: sizes where the decode and the large-tile kernel split K (the last slice shorter than the
others, columns that do not fill a tile, dropped and padding rows among the real ones), against the oracle; and the same
calls with a workspace that has no room for the slices' rows, which run uncut."""
import numpy as np
import pytest

from therock_amd import inputs as mi
from tests.test_gpu_fused_moe import check

# (tokens, experts, topk, hidden, inter, unit): decode kernel with one and with two token blocks, large tiles
DECODE = [(1, 4, 2, 64, 2176, 32), (5, 8, 3, 192, 1664, 64), (96, 4, 2, 320, 2176, 32)]
LARGE = [(171, 2, 2, 256, 2176, 32), (420, 2, 1, 384, 1664, 64)]
IDS = lambda s: "x".join(map(str, s))


def config(shape, dtype):
    T, E, K, H, I, unit = shape
    return mi.MoeConfig("slices", T, H, I, E, K, dtype, "softmax_renorm", unit=unit)


def needs(shape, dtype):
    """bytes of the workspace the library asks for"""
    import therock_amd as ta
    T, E, K, H, I, unit = shape
    traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, prec_o="fp16" if dtype == "fp16" else "bf16", block_m=unit)
    return ta.fused_moe_get_workspace_size(traits, T, E, K, H, I)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "int8", "fp8"])
@pytest.mark.parametrize("shape", DECODE + LARGE, ids=IDS)
def test_cut_down_gemm(shape, dtype, monkeypatch):
    import torch
    import therock_amd as ta
    cfg = config(shape, dtype)
    errs = [check(cfg, seed=3), check(cfg, seed=3, unfused=True)]
    rng = np.random.default_rng(5)
    check(cfg, seed=4, mask=(np.arange(cfg.experts) != rng.integers(cfg.experts)).astype(np.int32))
    check(cfg, seed=5, stride_pad=64)
    full = ta.MoeBuffers.__init__

    def short(self, *a, **kw):  # a workspace just too small for the cut
        full(self, *a, **kw)
        self.ws = torch.empty((self.ws.numel() - 256,), dtype=torch.uint8, device="cuda")

    monkeypatch.setattr(ta.MoeBuffers, "__init__", short)
    if needs(shape, dtype) > uncut(shape, dtype):
        errs.append(check(cfg, seed=3))
        assert errs[0] <= errs[-1] * 1.01  # fp32 shares: no further from the oracle than 16-bit partial rows


def uncut(shape, dtype):
    """The smallest workspace the call accepts (everything is checked on the host before anything is launched)."""
    import ctypes as C
    from therock_amd import _lib
    T, E, K, H, I, unit = shape
    lib = _lib.load()
    code = {"bf16": 0, "fp8": 1, "int8": 2}[dtype]
    t = _lib.FusedMoeTraits(code, code, 0, 3, 3, 3, 3, unit, 1, 0, 0, 0)
    f = _lib.FusedMoeArgs(block_m=unit, hidden_size=H, intermediate_size=I, num_tokens=T, num_experts=E, topk=K, stride_token=H)
    ws = _lib.Workspace(1 << 20, 0)  # an address that is never used: the null tensors are refused after the workspace
    lo, hi = 0, lib.mi355_fused_moe_workspace_size(C.byref(t), T, E, K, H, I) // 256
    while lo < hi:
        mid = (lo + hi) // 2
        ws.bytes = mid * 256
        if lib.mi355_fused_moe(C.byref(t), C.byref(f), C.byref(ws), None) == _lib.E_WORKSPACE:
            lo = mid + 1
        else:
            hi = mid
    return lo * 256


def test_workspace_without_room_for_the_slices_is_accepted():
    """The reported size has room for the slices' rows; what was enough without them still is (host side only)."""
    grown = 0
    for dtype in ("bf16", "int8", "fp8"):
        for shape in DECODE + LARGE:
            T, E, K, H, I, unit = shape
            rows = T * K + E * unit - K
            assert uncut(shape, dtype) <= needs(shape, dtype)
            grown += needs(shape, dtype) > uncut(shape, dtype)
            assert uncut(shape, dtype) >= rows * (H * 2 + I)  # partial rows and intermediate activations
    assert grown > 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp16", "int8", "fp8"])
@pytest.mark.parametrize("shape", DECODE + LARGE, ids=IDS)
def test_cut_stand_alone_down_gemm(shape, kind):
    from tests.test_gpu_moe_flatmm import test_gate_up_then_down as gate_up_then_down
    gate_up_then_down(*shape, kind)
