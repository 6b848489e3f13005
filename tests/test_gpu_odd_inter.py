"""int8 layers whose intermediate size is an odd multiple of 64 through the large-tile down GEMM, with bf16 and with re-quantised
int8 intermediate activations: rows of three weight pieces (the fewest whose last window is a half one that begins in another),
down GEMMs cut along K with last slices of one and of several pieces, both weight layouts, against plain fp32 products."""
import pytest

from therock_amd import inputs as mi
from tests.test_gpu_narrow_layers import rows

# (tokens, experts, topk, hidden, inter, unit), slices of K
SHAPES = [((420, 2, 1, 256, 192, 16), 1), ((420, 2, 1, 256, 320, 16), 1), ((700, 3, 2, 256, 448, 16), 1), ((700, 2, 2, 384, 832, 32), 2),
          ((420, 2, 1, 256, 1088, 16), 3), ((171, 2, 2, 128, 3264, 32), 7), ((1301, 2, 1, 256, 1600, 16), 4)]


def test_the_large_tiles_take_them():
    import therock_amd as ta
    for (T, E, K, H, I, unit), slices in SHAPES:
        assert rows("int8", T, E, K, H, I, unit) == 320
        for fq in (0, 2):
            traits = ta.fused_moe_traits(prec_i="int8", prec_w="int8", block_m=unit, fused_quant=fq)
            assert ta.fused_moe_k_slices(traits, T, E, K, H, I, 1 << 40) == slices
    assert rows("int8", 420, 2, 1, 256, 64, 16) != 320  # one piece: its window would begin before the weights


def test_waits_of_the_pipelined_loop(tmp_path):
    import os
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not installed")
    here = os.path.dirname(os.path.abspath(__file__))
    exe = tmp_path / "pipelined_schedule_check"
    subprocess.run([hipcc, "-std=c++17", "--cuda-host-only", "-I/opt/rocm/include", "-Wno-everything", "-o", str(exe),
                    os.path.join(here, "cpp", "pipelined_schedule_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and "pipelined_schedule_check ok" in r.stdout, r.stdout[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("fused_quant", [0, 2])
@pytest.mark.parametrize("shape", [s for s, _ in SHAPES], ids=lambda s: "x".join(map(str, s)))
def test_odd_inter(shape, fused_quant):
    import numpy as np
    import torch
    from tests.gpu_reference import fused_moe_fp32
    from tests.gpu_util import TORCH_DT, dev, run_fused_moe
    T, E, K, H, I, unit = shape
    cfg = mi.MoeConfig("odd", T, H, I, E, K, "int8", "softmax_renorm", unit=unit)
    inp = mi.make_inputs_np(cfg, 3)
    on = {k: None if v is None else dev(v) for k, v in inp.items()}
    for k in ("a", "g", "d"):
        on[k] = on[k].view(TORCH_DT["int8"])
    ref = fused_moe_fp32(cfg, on)
    plain, _ = run_fused_moe(cfg, inp, fused_quant=fused_quant)
    got = torch.from_numpy(plain.astype(np.int16)).cuda().view(torch.bfloat16).float()
    err = float((got - ref).norm() / ref.norm())
    print(f"odd {cfg} {fused_quant}: rel-L2 = {err:.3e}", flush=True)
    assert err <= (3e-2 if fused_quant else 1e-2)  # (as in the oracle tests: int8 intermediate rows with one scale each, or bf16)
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-30)
    assert float(per_row.max()) <= 6e-2  # a wrong step or window would show in whole rows
    shuffled, _ = run_fused_moe(cfg, inp, weight_permute=1, fused_quant=fused_quant)
    assert np.array_equal(plain, shuffled)
