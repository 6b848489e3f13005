"""Large tiles whose column tiles begin K at different places: which layers do is a matter of sizes, not of routing, and the
GEMMs that do (both of them, where weight rows lie whole 4 KiB apart) against plain fp32 products, cut along K and not, in
both weight layouts."""
import numpy as np
import pytest

from therock_amd import inputs as mi

# (dtype, fused_quant), (tokens, experts, hidden, inter), slices of the down GEMM
TYPES = [("bf16", 0), ("fp16", 0), ("fp8", 0), ("fp8", 2), ("int8", 0), ("int8", 2)]
CUT = (1600, 8, 512, 4096)
WHOLE = {2: (4000, 20, 2048, 2048), 1: (4000, 20, 2048, 4096)}


def elem(dtype):
    return 2 if dtype in ("bf16", "fp16") else 1


def traits(dtype, fq, permuted=0):
    import therock_amd as ta
    return ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, prec_o="fp16" if dtype == "fp16" else "bf16", block_m=32, fused_quant=fq,
                               weight_permute=permuted)


def test_the_large_tiles_take_them():
    import therock_amd as ta
    for dtype, fq in TYPES:
        for T, E, H, I in (CUT, WHOLE[elem(dtype)], (1200, 8, 4096, 4096)):
            assert I * elem(dtype) % 4096 == 0 and T // E <= 256
            assert ta.fused_moe_tile_rows(traits(dtype, fq), T, E, 1, H, I) == 320
            assert (ta.fused_moe_k_slices(traits(dtype, fq), T, E, 1, H, I, 1 << 40) == 1) == (E == 20)


def inputs(dtype, T, E, H, I, seed):
    import torch
    cfg = mi.MoeConfig("order", T, H, I, E, 1, dtype, "softmax_renorm")
    inp = mi.make_inputs_torch(cfg.scaled(dtype="bf16" if dtype == "fp16" else dtype), "cuda", seed)
    if dtype == "fp16":
        for k in ("a", "g", "d"):
            inp[k] = inp[k].to(torch.float16)
    return cfg, inp


def run(dtype, fq, cfg, inp, permuted=0):
    import torch
    import therock_amd as ta
    t = traits(dtype, fq, permuted)
    buf = ta.MoeBuffers(t, cfg.tokens, cfg.experts, 1, cfg.hidden, cfg.inter, "cuda")
    g, d = (ta.permute_weights(inp["g"]), ta.permute_weights(inp["d"])) if permuted else (inp["g"], inp["d"])
    args = ta.make_args(t, buf, inp["a"], g, d, inp["topk_ids"], inp["topk_weight"], a_scale=inp["a_scale"], g_scale=inp["g_scale"],
                        d_scale=inp["d_scale"])
    assert ta.fused_moe(t, args) == 0.0
    torch.cuda.synchronize()
    return buf.out


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,fq", TYPES)
def test_bits_do_not_depend_on_other_tokens_routing(dtype, fq):
    """320 tokens of an expert, alone (one row tile) and with one more (two): the same bits."""
    import torch
    T, E = 1200, 8
    cfg, inp = inputs(dtype, T, E, 4096, 4096, 3)
    ids = np.concatenate([np.zeros(320), 1 + np.arange(T - 320) % (E - 1)]).astype(np.int32)
    out = []
    for extra in (0, 1):
        ids[320] = 1 - extra
        inp["topk_ids"] = torch.from_numpy(ids.reshape(T, 1)).cuda()
        print(f"order {dtype} fused_quant={fq} rows={int((ids == 0).sum())}", flush=True)
        out.append(run(dtype, fq, cfg, inp)[:320].view(torch.int16).clone())
    assert torch.equal(out[0], out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("cut", [True, False])
@pytest.mark.parametrize("dtype,fq", TYPES)
def test_gemms_that_begin_elsewhere(dtype, fq, cut):
    import torch
    from tests.gpu_reference import fused_moe_fp32
    cfg, inp = inputs(dtype, *(CUT if cut else WHOLE[elem(dtype)]), 5)
    print(f"order {cfg} fused_quant={fq}", flush=True)
    ref = fused_moe_fp32(cfg, inp)
    plain = run(dtype, fq, cfg, inp)
    got = plain.float()
    err = float((got - ref).norm() / ref.norm())
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-30)
    print(f"  rel-L2 = {err:.3e}, worst row {float(per_row.max()):.3e}", flush=True)
    # as in the oracle tests: 8-bit intermediate activations, or 16-bit ones; a window taken twice or left out would show in
    # whole rows (one of 32 or 64 windows is an eighth to a sixth of a row's norm)
    assert err <= (3e-2 if dtype == "fp8" or fq else 1e-2) and float(per_row.max()) <= 8e-2
    assert torch.equal(plain.view(torch.int16), run(dtype, fq, cfg, inp, permuted=1).view(torch.int16))
