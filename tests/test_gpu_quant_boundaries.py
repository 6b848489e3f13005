"""Activation quantisers at the quotients where codes change: the kernels bracket a quotient in fp32 and fall back to the
exactly rounded one where the bracket's ends disagree, so values next to every code boundary, and scales outside the
bracket's range, have to give the oracle's bytes."""
import os
import re

import numpy as np
import pytest

import oracle

E4M3_STEPS = [m * 2.0 ** e for e in range(-10, 9) for m in np.arange(8, 16, 0.5) / 8] + [k * 2.0 ** -10 for k in range(1, 17)]


def boundary_rows(kind, exponents, hidden, seed):
    """fp32 rows of quotients at, and one to three ulps beside, the boundaries of every code, for row maxima 2^exponent."""
    rng = np.random.default_rng(seed)
    qmax = np.float32(127 if kind == "int8" else 448)
    steps = np.arange(0, 127.25, 0.5) if kind == "int8" else np.array([v for v in E4M3_STEPS if v <= 448])
    rows = []
    for e in exponents:
        amax = np.float32((1 + rng.random()) * 2.0 ** e)
        v = (steps * np.float64(amax / qmax)).astype(np.float32)
        near = np.concatenate([v] + [(v.view(np.int32) + d).clip(0).view(np.float32) for d in (-3, -2, -1, 1, 2, 3)])
        near = rng.permutation(np.minimum(near, amax))
        row = np.resize(near, hidden) * rng.choice(np.float32([-1, 1]), hidden)
        row[rng.integers(hidden)] = amax
        rows.append(row)
    return np.stack(rows)


def e4m3_codes(q):
    import torch
    return torch.from_numpy(np.ascontiguousarray(q, np.float32)).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).numpy()


def codes_of(q, kind):
    return np.clip(np.trunc(q), -127, 127).astype(np.int8) if kind == "int8" else e4m3_codes(q)


def bracket(v, amax, kind, ulp):
    """Both ends of the bracket of v / (amax / qmax), with the hardware reciprocal `ulp` ulps off and the kernels' margins."""
    src = open(os.path.join(os.path.dirname(os.path.dirname(__file__)), "therock_amd", "csrc", "moe_quant.hip")).read()
    margins = [float(sign + str(2.0 ** -int(e))) for sign, e in re.findall(r"= r \* \(1\.0f ([+-]) 0x1p-(\d+)f\);", src.replace("  ", ""))]
    assert len(margins) == 2 and margins[0] < 0 < margins[1]
    qmax = np.float32(127 if kind == "int8" else 448)
    r = (1 / amax.astype(np.float64)).astype(np.float32)
    r = qmax * (r.view(np.int32) + ulp).view(np.float32)
    return [v * (r * np.float32(1 + m)) for m in margins]


@pytest.mark.parametrize("ulp", [-1, 0, 1])
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_bracket_encloses_the_division(kind, ulp):
    """On the CPU, over the range of row maxima the kernels bracket: the fp32 division lies between the ends, and where both
    give one code it is the division's."""
    qmax = np.float32(127 if kind == "int8" else 448)
    v = boundary_rows(kind, range(-99, 100, 6), 4096, 5)
    amax = np.abs(v).max(axis=1, keepdims=True)
    q = v / (amax / qmax)
    lo, hi = bracket(v, amax, kind, ulp)
    normal = np.abs(q) >= 2.0 ** -100
    assert (np.where(normal, np.abs(lo) <= np.abs(q), True)).all() and (np.where(normal, np.abs(q) <= np.abs(hi), True)).all()
    codes, agree = codes_of(q, kind), codes_of(lo, kind) == codes_of(hi, kind)
    assert np.array_equal(codes[agree], codes_of(lo, kind)[agree])
    assert 0.3 < agree.mean() < 0.9  # both outcomes are met: values beside a boundary, and those in a code's middle


# rows of one, two and four pieces a thread and longer ones; tables that stay in L2 and that do not
@pytest.mark.gpu
@pytest.mark.parametrize("hidden,experts", [(1864, 8), (4096, 8), (4096, 256), (4104, 8), (8192, 128), (8200, 8), (10240, 96)])
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_smoothquant_codes_at_boundaries(hidden, experts, kind):
    import torch
    import therock_amd as ta

    exponents = np.resize([0, -30, 40, -99, 99, -101, 101, -120, 120], experts)
    sm = boundary_rows(kind, exponents, hidden, hidden + experts)
    tokens = 2 * experts
    x = torch.ones((tokens, hidden), dtype=torch.bfloat16, device="cuda")
    ids = np.stack([(np.arange(2) * 3 + t) % experts for t in range(tokens)]).astype(np.int32)
    qy, ys = ta.moe_smoothquant(x, torch.from_numpy(sm).cuda(), torch.from_numpy(ids).cuda(), kind)
    torch.cuda.synchronize()
    rq, rs = oracle.smoothquant(np.ones((tokens, hidden), np.float32), sm, ids, oracle.DT_I8 if kind == "int8" else oracle.DT_E4M3)
    assert np.array_equal(ys.cpu().numpy(), rs)
    assert np.array_equal(qy.view(torch.uint8).cpu().numpy(), rq.view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("fq", [1, 2])
@pytest.mark.parametrize("dtype", ["int8", "fp8"])
@pytest.mark.parametrize("inter", [2048, 2176, 4224])
def test_requantised_rows_around_a_lanes_registers(inter, dtype, fq):
    # up to 2048 columns a lane keeps its pieces and codes come from the bracket; longer rows take the exact quotients
    from therock_amd import inputs as mi
    from tests.test_gpu_fused_quant import run
    run(mi.MoeConfig("fq_long_rows", 48, 256, inter, 4, 2, dtype, "softmax_renorm"), fq)


# ---- codes between the GEMMs.  Token t goes to expert t with weight 1; the intermediate activations are set value by value
# through the scales (silu(64) is 64 in fp32), and down weights of the identity bring every code, times its row's scale, to
# the output, where neighbouring codes stay apart: c * scale in bf16, c of up to 7 bits.
def bf16_rows(kind, exponents, cols, seed):
    """Like boundary_rows, of values that bf16 holds (exact ties where the maximum is qmax times a power of two)."""
    import torch
    rng = np.random.default_rng(seed)
    qmax = 127 if kind == "int8" else 448
    steps = np.arange(0, 127.25, 0.5) if kind == "int8" else np.array([v for v in E4M3_STEPS if v <= 448])
    rows = []
    for n, e in enumerate(exponents):
        amax = np.float32((qmax / 128 if n % 2 == 0 else (128 + rng.integers(128)) / 128) * 2.0 ** e)
        v = torch.from_numpy((steps * np.float64(amax) / qmax).astype(np.float32)).to(torch.bfloat16).view(torch.int16)
        near = np.concatenate([(v + d).clamp(min=0).view(torch.bfloat16).float().numpy() for d in (-1, 0, 1)])
        row = np.resize(rng.permutation(np.minimum(near, amax)), cols) * rng.choice(np.float32([-1, 1]), cols)
        row[rng.integers(cols)] = amax
        rows.append(row)
    return np.stack(rows)


@pytest.mark.gpu
@pytest.mark.parametrize("fq", [1, 2])
@pytest.mark.parametrize("dtype", ["int8", "fp8"])
# (a row to a wave up to 2048 columns, to 256 threads up to 8192, to 512 beyond, which hold 16384 columns of it)
@pytest.mark.parametrize("inter", [512, 2048, 2176, 4224, 8192, 8320, 16384, 16512])
def test_requantised_codes_at_boundaries(inter, dtype, fq):
    import torch
    import therock_amd as ta
    exponents = [0, 0, -30, 40, -99, 98, -101, 101, 112, 112]  # (the least value, 2^-19 of the maximum / 64, stays normal)
    v = (boundary_rows if fq == 1 else bf16_rows)(dtype, exponents, inter, inter + fq)
    v = np.concatenate([v, np.zeros((1, inter), np.float32)])  # a row of zeros
    E = T = len(v)
    print(f"requantised codes {dtype} fused_quant={fq} inter={inter}", flush=True)
    st, one = (torch.int8, 1) if dtype == "int8" else (torch.uint8, 0x38)
    view = torch.int8 if dtype == "int8" else torch.float8_e4m3fn
    H = inter
    a = torch.zeros((T, H), dtype=st, device="cuda")
    g = torch.zeros((E, (2 if fq == 2 else 1) * inter, H), dtype=st, device="cuda")
    d = torch.zeros((E, H, inter), dtype=st, device="cuda")
    a[:, 0], g[:, :, 0] = one, one
    d.diagonal(dim1=1, dim2=2).fill_(one)
    g_scale = torch.ones(g.shape[:2], dtype=torch.float32, device="cuda")
    values = torch.from_numpy(v).cuda()
    smooth = None
    if fq == 1:  # gate only: every activation is 64, the smooth scale makes the value of it
        smooth = (values / 64).contiguous()
    else:
        g_scale[:, inter:] = values / 4096  # 64 of the gate half, 64 of the tokens' scale
    traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, block_m=32, gate_only=int(fq == 1), fused_quant=fq)
    buf = ta.MoeBuffers(traits, T, E, 1, H, inter, "cuda")
    args = ta.make_args(traits, buf, a.view(view), g.view(view), d.view(view), torch.arange(T, dtype=torch.int32, device="cuda").reshape(T, 1),
                        torch.ones((T, 1), device="cuda"), a_scale=torch.full((T,), 64.0, device="cuda"), g_scale=g_scale,
                        d_scale=torch.ones((E, H), device="cuda"))
    args.y_smooth_scale_ptr = smooth
    assert ta.fused_moe(traits, args) == 0.0
    torch.cuda.synchronize()

    amax = np.abs(v).max(axis=1, keepdims=True)
    scale = amax / np.float32(127 if dtype == "int8" else 448)
    q = v / np.where(amax > 0, scale, np.float32(1))
    codes = np.rint(q) if dtype == "int8" else oracle.e4m3_to_f32(e4m3_codes(q))
    want = torch.from_numpy(codes.astype(np.float32) * scale).to(torch.bfloat16)
    got = buf.out.cpu()
    assert torch.equal(got.float(), want.float()), int((got.float() != want.float()).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_rows_with_nan_and_infinity(kind):
    """The same row in both forms of the kernels, 4096 columns from the bracket and longer (zeros behind) from the exact
    quotients: the same bytes."""
    import torch
    import therock_amd as ta
    rng = np.random.default_rng(2)
    x = rng.standard_normal((8, 4096)).astype(np.float32)
    x[0, rng.integers(0, 4096, 40)] = np.nan
    x[1, 77], x[2, 4095] = np.inf, -np.inf
    x[3, 5], x[3, 900:1100] = -np.inf, np.nan
    x[4] = np.nan
    x[5] *= 2.0 ** 124
    x[6] *= 2.0 ** -130
    x[7, ::2] = np.nan
    short = torch.from_numpy(x).to(torch.bfloat16).cuda()
    long = torch.zeros((8, 4608), dtype=torch.bfloat16, device="cuda")
    long[:, :4096] = short
    ids = torch.zeros((8, 1), dtype=torch.int32, device="cuda")
    sm = torch.ones((2, 4608), dtype=torch.float32, device="cuda")
    for f in (lambda r: ta.rowwise_quant(r, kind), lambda r: ta.moe_smoothquant(r, sm[:, :r.shape[1]].contiguous(), ids, kind)):
        (q, s), (ql, sl) = f(short), f(long)
        torch.cuda.synchronize()
        assert torch.equal(s.view(torch.int32), sl.view(torch.int32))
        assert torch.equal(q.view(torch.uint8), ql.view(torch.uint8)[..., :4096])
