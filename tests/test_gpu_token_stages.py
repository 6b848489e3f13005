"""The large-tile kernel's token stages, whose number depends on the rows of a tile: one batch holds tiles of one to five 64-row
groups, over K of two steps (fewer than there are stages) up to a few rounds of the stages, and with 8-bit operands over odd
step counts, where the half last window goes out ahead of the loop or inside it; against plain fp32 products."""
import numpy as np
import pytest

from therock_amd import inputs as mi
from tests.test_gpu_narrow_layers import rows

COUNTS = (30, 100, 170, 250, 310, 441)  # rows per expert: 1, 2, 3, 4, 5 and twice 4 groups
ODD = (60, 101, 170, 471)               # 1, 2, 3 and twice 4 groups
# (dtype, hidden, inter, rows per expert)
CASES = [("bf16", h, i, COUNTS) for h, i in ((64, 64), (192, 128), (448, 320), (960, 512))]
CASES += [("int8", h, i, COUNTS) for h, i in ((128, 128), (384, 192), (896, 448))]
CASES += [("fp8", h, i, COUNTS) for h, i in ((128, 128), (384, 256), (896, 512))]
CASES += [(t, h, i, ODD) for t in ("int8", "fp8") for h, i in ((320, 13184), (448, 9472), (576, 7424), (704, 6016))]


def test_the_large_tiles_take_them():
    for dtype, H, I, counts in CASES:
        assert rows(dtype, sum(counts), len(counts), 1, H, I, 16) == 320


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:3])))
def test_token_stages(case):
    import torch
    from tests.gpu_reference import fused_moe_fp32
    from tests.gpu_util import TORCH_DT, dev, run_fused_moe
    dtype, H, I, counts = case
    cfg = mi.MoeConfig("stages", sum(counts), H, I, len(counts), 1, dtype, "softmax_renorm", unit=16)
    inp = mi.make_inputs_np(cfg, 7)
    ids = np.repeat(np.arange(len(counts)), counts).astype(np.int32)
    inp["topk_ids"] = np.random.default_rng(1).permutation(ids).reshape(-1, 1)
    on = {k: None if v is None else dev(v) for k, v in inp.items()}
    for k in ("a", "g", "d"):
        on[k] = on[k].view(TORCH_DT[dtype])
    ref = fused_moe_fp32(cfg, on)
    plain, _ = run_fused_moe(cfg, inp)
    got = torch.from_numpy(plain.astype(np.int16)).cuda().view(torch.bfloat16).float()
    err = float((got - ref).norm() / ref.norm())
    print(f"stages {case}: rel-L2 = {err:.3e}", flush=True)
    assert err <= (3e-2 if dtype == "fp8" else 1e-2)  # fp8: intermediate activations are e4m3 as well (as in the oracle tests)
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-30)
    assert float(per_row.max()) <= 8e-2  # a stage overwritten or read early would show in whole rows
    again, _ = run_fused_moe(cfg, inp, weight_permute=1)
    assert np.array_equal(plain, again)
