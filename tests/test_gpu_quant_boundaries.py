"""Activation quantisers at the quotients where codes change: the kernels bracket a quotient in fp32 and fall back to the
exactly rounded one where the bracket's ends disagree, so values next to every code boundary, and scales outside the
bracket's range, have to give the oracle's bytes."""
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


def bracket_codes(v, amax, kind, ulp):
    """Codes from both ends of the bracket of v / (amax / qmax), with the hardware reciprocal `ulp` ulps off."""
    qmax = np.float32(127 if kind == "int8" else 448)
    r = (1 / amax.astype(np.float64)).astype(np.float32)
    r = qmax * (r.view(np.int32) + ulp).view(np.float32)
    ends = [v * (r * np.float32(1 + s * 2.0 ** -20)) for s in (-1, 1)]
    return [np.clip(np.trunc(q), -127, 127) if kind == "int8" else q for q in ends]


@pytest.mark.parametrize("ulp", [-1, 0, 1])
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_bracket_encloses_the_division(kind, ulp):
    """On the CPU, over the range of row maxima the kernels bracket: the fp32 division lies between the ends, hence (int8,
    toward zero) its code between theirs."""
    qmax = np.float32(127 if kind == "int8" else 448)
    v = boundary_rows(kind, range(-99, 100, 6), 4096, 5)
    amax = np.abs(v).max(axis=1, keepdims=True)
    q = v / (amax / qmax)
    lo, hi = bracket_codes(v, amax, kind, ulp)
    if kind == "int8":
        q = np.trunc(q)
    normal = np.abs(q) >= 2.0 ** -100
    assert (np.where(normal, np.abs(lo) <= np.abs(q), True)).all() and (np.where(normal, np.abs(q) <= np.abs(hi), True)).all()
    assert (lo == hi).mean() > 0.3 if kind == "int8" else True


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
