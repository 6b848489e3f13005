"""The work a user of the fused-MoE path has it do, as cases that can be timed and compared.

A case is one pass of a mixture-of-experts layer over one batch, in one of the three ways the public entry points are
put together:

  "layer"   router (topk_softmax) -> per-token quantisation of the activations (8-bit types) -> fused_moe
  "smooth"  router -> moe_smoothquant -> fused_moe with fused_quant 1 (smooth-quantised int8 / fp8 models)
  "gemms"   router -> moe_sorting (which also clears the output) -> moe_flatmm gate+up -> moe_flatmm down (layers with
            expert biases and the clamped SwiGLU, which keep the two GEMMs apart)

What a serving program has in hand before the pass is made by prepare(): weights (quantised once, at load time), hidden
states and router logits of the batch, and the buffers it keeps.  Batches run from one decoding sequence to a long
prefill; the models are the ones the benchmark and the tests of this repository use, and generic ones like them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import therock_amd as ta
from therock_amd.inputs import zipf_bias

ELEM_BYTES = {"bf16": 2, "fp16": 2, "fp8": 1, "int8": 1}
TORCH_TYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.float8_e4m3fn, "int8": torch.int8}

# every field a case can have; listed() and draw() state what differs
DEFAULTS = {
    "kind": "layer", "dtype": "bf16", "tokens": 1, "hidden": 1024, "inter": 1024, "experts": 8, "topk": 2,
    "router": "softmax",      # softmax | sigmoid: what turns the logits into weights
    "renorm": True,           # weights of a token add up to one
    "skew": False,            # logits biased so that experts are chosen with Zipf frequencies
    "block_m": 32,            # unit of the sort
    "activation": 1,          # 1 silu, 0 gelu
    "gate_only": 0,
    "fused_quant": 0,         # 2: intermediate activations re-quantised per row ("smooth" runs with 1)
    "preshuffled": False,     # weights kept in ck_tile's b_nr_kr_kw_nw_kv layout
    "local_experts": 0,       # expert parallelism: this rank owns the first so many experts (0: all of them)
}


def _case(name=None, **kw):
    assert set(kw) <= set(DEFAULTS)
    c = dict(DEFAULTS, **kw)
    return c if name is None else {"name": name, **c}


SMALL = dict(hidden=1024, inter=1024, experts=8, topk=2)                  # the layer a CPU reference can run
WIDE = dict(hidden=4096, inter=14336, experts=8, topk=2)                  # few wide experts
FINE = dict(hidden=7168, inter=2048, experts=256, topk=8, router="sigmoid")  # many narrow ones
MEDIUM = dict(hidden=4096, inter=1536, experts=128, topk=8, renorm=False)
SKEWED = dict(hidden=2048, inter=1408, experts=64, topk=6, skew=True)
BIASED = dict(hidden=2880, inter=2880, experts=32, topk=4)


def listed():
    return [
        # one sequence decoding on a small layer: launches and host work are all there is
        _case("one token bf16", tokens=1, **SMALL),
        # the same layer with a modest batch
        _case("small batch bf16", tokens=128, **SMALL),
        # a serving batch decoding: every expert's weights are streamed for a handful of rows
        _case("decode int8", dtype="int8", tokens=64, **MEDIUM),
        # the same with popular experts (Zipf routing): few experts with many rows
        _case("decode int8 skewed", dtype="int8", tokens=256, skew=True, **MEDIUM),
        # decoding with many experts of which a third is idle in a batch
        _case("decode fp8", dtype="fp8", tokens=13, **FINE),
        # between decode and prefill: a short chunk, ragged rows per expert
        _case("chunk bf16", tokens=333, **WIDE),
        _case("chunk fp8", dtype="fp8", tokens=1000, **FINE),
        # prefill
        _case("prefill fp8", dtype="fp8", tokens=8192, **FINE),
        _case("prefill bf16 preshuffled", tokens=4096, preshuffled=True, **WIDE),
        _case("prefill bf16 skewed", tokens=32768, **SKEWED),
        # a smooth-quantised int8 model, activations quantised once per (token, expert)
        _case("prefill int8 smooth", kind="smooth", dtype="int8", tokens=3001, **MEDIUM),
        # a layer with expert biases and clamped SwiGLU, run as two stand-alone GEMMs
        _case("gemms fp16 biased", kind="gemms", dtype="fp16", tokens=777, **BIASED),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: batches of 1 .. 32768 tokens, layers of 4 .. 256 experts, hidden and
    intermediate sizes of the models above and odd ones between them, every operand type and option."""
    kind = rng.choice(["layer"] * 6 + ["smooth", "gemms"])
    dtype = rng.choice(["int8", "fp8"] if kind == "smooth" else ["bf16", "fp16", "fp8", "int8"] if kind == "layer" else ["bf16", "fp16"])
    c = _case(kind=kind, dtype=dtype)
    c["experts"] = _log_int(rng, 4, 256)
    c["topk"] = min(rng.randint(1, 8), c["experts"] // 2)
    c["hidden"] = 64 * _log_int(rng, 8, 112)       # 512 .. 7168
    step = 128 if dtype == "fp8" else 64
    c["inter"] = step * _log_int(rng, 512 // step, 14336 // step)
    c["tokens"] = _log_int(rng, 1, 32768)
    c["router"] = rng.choice(["softmax", "sigmoid"])
    c["renorm"] = rng.random() < 0.7
    c["skew"] = rng.random() < 0.3
    c["block_m"] = rng.choice([32, 32, 32, 64])
    if kind == "layer":
        option = rng.choice(["none", "none", "none", "preshuffled", "gelu", "gate_only", "local", "quant"])
        if option == "preshuffled":
            c["preshuffled"] = True
        elif option == "gelu":
            c["activation"] = 0
        elif option == "gate_only":
            c["gate_only"] = 1
        elif option == "local":
            c["local_experts"] = max(1, c["experts"] // rng.choice([2, 4]))
        elif option == "quant" and dtype in ("fp8", "int8"):
            c["fused_quant"] = 2
    # no more weights and no more work than the largest listed cases
    b = ELEM_BYTES[dtype]
    while 3 * c["experts"] * c["hidden"] * c["inter"] * b > 8e9:
        c["experts"] = max(4, c["experts"] // 2)
        c["inter"] = c["inter"] if c["experts"] > 4 else max(step, c["inter"] // 2 // step * step)
    c["topk"] = min(c["topk"], c["experts"] // 2)
    c["local_experts"] = min(c["local_experts"], c["experts"] // 2)
    most = 4e12 / (6.0 * c["topk"] * c["hidden"] * c["inter"] * b)
    c["tokens"] = max(1, min(c["tokens"], int(most), int(1.5e9 / (c["topk"] * max(c["hidden"], c["inter"]) * 2))))
    return c


# ------------------------------------------------------------------------------------------------ preparation
def _weights(gen, case, n, k, count):
    """[count, n, k] weights N(0, 0.02), and per-row scales for the 8-bit types."""
    st = TORCH_TYPE[case["dtype"]]
    w = torch.empty((count, n, k), dtype=st, device="cuda")
    quant = ELEM_BYTES[case["dtype"]] == 1
    s = torch.empty((count, n), dtype=torch.float32, device="cuda") if quant else None
    chunk = max(1, min(count, (1 << 28) // (n * k)))
    for e0 in range(0, count, chunk):
        e1 = min(count, e0 + chunk)
        v = torch.randn((e1 - e0, n, k), generator=gen, device="cuda") * 0.02
        if quant:
            qmax = 448.0 if case["dtype"] == "fp8" else 127.0
            s[e0:e1] = v.abs().amax(dim=-1).clamp_(min=1e-20) / qmax
            v /= s[e0:e1, :, None]
            if case["dtype"] == "int8":
                v.round_()
            v.clamp_(-qmax, qmax)
        w[e0:e1] = v.to(st)
    return w, s


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "topk"))
    own = case["local_experts"] or E
    st = {"case": case}
    # hidden states arrive as bf16 (fp16 for an fp16 model), router logits as fp32
    st["x"] = torch.randn((T, H), generator=gen, device="cuda").to(torch.float16 if case["dtype"] == "fp16" else torch.bfloat16)
    logits = torch.randn((T, E), generator=gen, device="cuda")
    if case["skew"]:
        logits += torch.from_numpy(zipf_bias(E)).to("cuda")
    st["logits"] = logits
    st["g"], st["g_scale"] = _weights(gen, case, I if case["gate_only"] else 2 * I, H, own)
    st["d"], st["d_scale"] = _weights(gen, case, H, I, own)
    if case["preshuffled"]:
        st["g"], st["d"] = ta.permute_weights(st["g"]), ta.permute_weights(st["d"])
    if case["kind"] == "gemms":
        unit, out = case["block_m"], TORCH_TYPE[case["dtype"]]
        n = ta.moe_max_num_tokens_padded(T, E, K, unit)
        st["sorted_ids"] = torch.empty((n,), dtype=torch.int32, device="cuda")
        st["sorted_w"] = torch.empty((n,), dtype=torch.float32, device="cuda")
        st["sorted_eid"] = torch.empty((-(-n // unit),), dtype=torch.int32, device="cuda")
        st["total"] = torch.empty((2,), dtype=torch.int32, device="cuda")
        st["g_bias"] = torch.randn((E, 2 * I), generator=gen, device="cuda") * 0.1
        st["d_bias"] = torch.randn((E, H), generator=gen, device="cuda") * 0.1
        st["y"] = torch.empty((T * K, I), dtype=out, device="cuda")
        st["out"] = torch.empty((T, H), dtype=out, device="cuda")
        st["sort_ws"] = torch.empty((max(ta.moe_sorting_get_workspace_size(T, E, K), 256),), dtype=torch.uint8, device="cuda")
        ws = max(ta.moe_flatmm_get_workspace_size(ta.GEMM1_GATE_UP, st["x"], st["g"], st["y"], st["sorted_ids"], st["sorted_eid"], st["total"], T, K, unit),
                 ta.moe_flatmm_get_workspace_size(ta.GEMM2, st["y"], st["d"], st["out"], st["sorted_ids"], st["sorted_eid"], st["total"], T, K, unit))
        st["ws"] = torch.empty((max(ws, 256),), dtype=torch.uint8, device="cuda")
        return st
    st["traits"] = ta.fused_moe_traits(
        prec_i=case["dtype"], prec_w=case["dtype"], prec_o="fp16" if case["dtype"] == "fp16" else "bf16", block_m=case["block_m"],
        activation=case["activation"], gate_only=case["gate_only"], fused_quant=1 if case["kind"] == "smooth" else case["fused_quant"],
        local_expert_masking=bool(case["local_experts"]), weight_permute=int(case["preshuffled"]))
    st["buf"] = ta.MoeBuffers(st["traits"], T, E, K, H, I, "cuda")
    st["mask"] = None
    if case["local_experts"]:
        st["mask"] = (torch.arange(E, device="cuda") < own).to(torch.int32)
    if case["kind"] == "smooth":
        st["x_smooth"] = torch.rand((E, H), generator=gen, device="cuda") + 0.5
        st["y_smooth"] = torch.rand((E, I), generator=gen, device="cuda") + 0.5
        st["qx"] = (torch.empty((K, T, H), dtype=TORCH_TYPE[case["dtype"]], device="cuda"), torch.empty((K, T), dtype=torch.float32, device="cuda"))
    return st


# ------------------------------------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    w, ids = ta.topk_softmax(st["logits"], case["topk"], activation=case["router"], renormalize=case["renorm"])
    if case["kind"] == "gemms":
        T, K, unit = case["tokens"], case["topk"], case["block_m"]
        ta.moe_sorting(ta.moe_sorting_trait(), ta.moe_sorting_args(
            p_topk_ids=ids, p_weights=w, p_sorted_token_ids=st["sorted_ids"], p_sorted_weights=st["sorted_w"],
            p_sorted_expert_ids=st["sorted_eid"], p_total_tokens_post_pad=st["total"], p_moe_buf=st["out"], p_ws=st["sort_ws"],
            tokens=T, unit_size=unit, num_experts=case["experts"], topk=K, moe_buf_interm_dim=case["hidden"],
            moe_buf_elem_bytes=st["out"].element_size()))
        ta.moe_flatmm(ta.GEMM1_GATE_UP, st["x"], st["g"], st["y"], st["sorted_ids"], st["sorted_eid"], st["total"], T, K, unit,
                      exp_bias=st["g_bias"], activation=ta.ACT_SWIGLU, workspace=st["ws"])
        ta.moe_flatmm(ta.GEMM2, st["y"], st["d"], st["out"], st["sorted_ids"], st["sorted_eid"], st["total"], T, K, unit,
                      sorted_weights=st["sorted_w"], exp_bias=st["d_bias"], workspace=st["ws"])
        return [st["out"], st["y"], w, ids]
    a, a_scale, smooth = st["x"], None, None
    if case["kind"] == "smooth":
        q, a_scale = ta.moe_smoothquant(st["x"], st["x_smooth"], ids, q_dtype=case["dtype"], out=st["qx"])
        a, smooth = q[0], st["y_smooth"]  # the rows of slot 0: the other slots' follow them in memory
    elif ELEM_BYTES[case["dtype"]] == 1:
        a, a_scale = ta.rowwise_quant(st["x"], case["dtype"])
    args = ta.make_args(st["traits"], st["buf"], a, st["g"], st["d"], ids, w, a_scale=a_scale, g_scale=st["g_scale"],
                        d_scale=st["d_scale"], local_expert_mask=st["mask"], num_experts=case["experts"])
    args.y_smooth_scale_ptr = smooth
    ta.fused_moe(st["traits"], args)
    return [st["buf"].out, w, ids]


# ------------------------------------------------------------------------------------------------ what a pass needs
def _experts_used(case):
    """Expected number of this rank's experts that at least one token of the batch chooses."""
    T, E, K = case["tokens"], case["experts"], case["topk"]
    rng = np.random.default_rng(0)
    n = 4096
    logits = rng.standard_normal((n, E)).astype(np.float32) + (zipf_bias(E) if case["skew"] else 0.0)
    p = np.bincount(np.argpartition(-logits, K - 1, axis=1)[:, :K].ravel(), minlength=E) / n
    return float(np.sum((1.0 - (1.0 - p) ** T)[:case["local_experts"] or E])), float(np.sum(p[:case["local_experts"] or E]) / K)


def work(case):
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "topk"))
    b = ELEM_BYTES[case["dtype"]]
    used, share = _experts_used(case)
    rows = 2 if case["gate_only"] else 3  # weight matrices of I x H per expert
    size = used * rows * H * I * b + T * H * 2 + T * E * 4 + T * H * 2 + T * K * 8
    if b == 1:
        size += used * ((rows - 1) * I + H) * 4
    if case["kind"] == "smooth":
        size += used * (H + I) * 4
    if case["kind"] == "gemms":
        size += used * (2 * I + H) * 4 + T * K * I * 2
    return {"bytes": size, "flops": 2.0 * rows * T * K * share * H * I}


def tolerance(case):
    """Results are 16-bit floats: an fp16 path keeps its intermediate results in fp16; with bf16 the intermediate
    activations, the partial rows and the output are each rounded to 8 bits; 8-bit models with 8-bit intermediate
    activations also see the codes that a last-bit difference moves to a neighbour.  Expert ids: near ties only."""
    if case["dtype"] == "fp16":
        rel = 1e-3
    else:
        rel = 5e-3 if case["dtype"] == "bf16" or (case["dtype"] == "int8" and case["kind"] == "layer" and not case["fused_quant"]) else 1e-2
    return {"rel": rel, "differ": 1e-4}
