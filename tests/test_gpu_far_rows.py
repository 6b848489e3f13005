"""Token rows so far apart that a 32-bit byte offset does not reach them all: such calls run without the large tiles and the
decode kernel, whatever height the sizes would have with packed rows, and with no second height for the sort to take."""
import ctypes as C

import numpy as np
import pytest

from therock_amd import _lib

FAR = 1 << 32  # bytes


def traits(dtype, fq=0):
    import therock_amd as ta
    return ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, block_m=32, fused_quant=fq)


# (dtype, fused_quant, tokens, experts, topk, hidden, inter, zipf): large tiles; large tiles, the down GEMM cut; smooth-quant
# rows per (slot, token); fp8 on decode tiles whose sort may take the large ones
FUSED = [("bf16", 0, 2048, 8, 2, 512, 384, 0), ("fp8", 0, 104, 5, 2, 512, 8576, 0), ("int8", 1, 640, 8, 2, 512, 448, 0),
         ("fp8", 0, 256, 64, 4, 512, 2048, 1)]


def pitch(dtype, rows):
    """Elements between rows that bring them to 4 GiB and a little more."""
    return -(-FAR // (rows * (1 if dtype != "bf16" else 2)) // 64) * 64 + 64


def test_sizes():
    """What these calls would run on with packed rows."""
    import therock_amd as ta
    for dtype, fq, T, E, K, H, I, zipf in FUSED:
        assert ta.fused_moe_tile_rows(traits(dtype, fq), T, E, K, H, I) == (32 if zipf else 320)
    t = traits("fp8").pod()
    T, E, K, H, I = FUSED[3][2:7]
    assert _lib.load().mi355_fused_moe_chosen_tile_rows(C.byref(t), T, E, K, H, I, None, None) == 0 # the sort's choice
    assert ta.fused_moe_k_slices(traits("fp8"), 104, 5, 2, 512, 8576, 1 << 40) == 6


def stand_alone(T, E, K, inter, hidden, stride):
    a = _lib.FlatmmArgs()
    a.NumTokens, a.NumExperts, a.TopK, a.N, a.K, a.block_m, a.k_batch = T, E, K, hidden, inter, 32, 1
    a.stride_A, a.stride_B, a.stride_C = stride, inter, hidden
    a.prec_a, a.prec_b = _lib.DTYPES["bf16"], _lib.DTYPES["int8"]
    return a


def test_far_rows_are_accepted():
    """Host side: past every check, with the workspace the library reports, a call fails only for want of a GPU."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("calls with made-up addresses: only where nothing can be launched")
    lib, at = _lib.load(), 1 << 20
    for dtype, fq, T, E, K, H, I, _ in FUSED:
        t = traits(dtype, fq).pod()
        need = lib.mi355_fused_moe_workspace_size(C.byref(t), T, E, K, H, I)
        for stride, size, want in ((pitch(dtype, T * (K if fq == 1 else 1)), need, _lib.E_HIP), (H, 0, _lib.E_WORKSPACE)):
            g = _lib.FusedMoeGemmArgs(hidden_size=H, intermediate_size=I, num_tokens=T, num_experts=E, topk=K, stride_token=stride)
            for f in ("a_ptr", "a_scale_ptr", "g_ptr", "d_ptr", "g_scale_ptr", "d_scale_ptr", "o_ptr", "sorted_token_ids_ptr",
                      "sorted_weight_ptr", "sorted_expert_ids_ptr", "num_sorted_tiles_ptr") + (("y_smooth_scale_ptr",) if fq == 1 else ()):
                setattr(g, f, at)
            ws = _lib.Workspace(at, size)
            assert lib.mi355_fused_moegemm(C.byref(t), C.byref(g), C.byref(ws), None) == want, (dtype, stride, lib.mi355_moe_last_error())
    a = stand_alone(20000, 8, 4, 1728, 512, 28000)
    for f in ("p_sorted_token_ids", "p_sorted_expert_weights", "p_sorted_expert_ids", "p_max_token_id", "a_ptr", "b_ptr", "c_ptr", "scale_n"):
        setattr(a, f, at)
    packed = stand_alone(20000, 8, 4, 1728, 512, 1728)
    need = lib.mi355_moe_flatmm_workspace_size(2, C.byref(a))
    assert need == lib.mi355_moe_flatmm_workspace_size(2, C.byref(packed))
    ws = _lib.Workspace(at, need)
    assert lib.mi355_moe_flatmm(2, C.byref(a), C.byref(ws), None) == _lib.E_HIP, lib.mi355_moe_last_error()


def test_library_workspace_holds_what_it_held():
    """The list's room for far rows does not push a call over the library-owned workspace: layers that fill 96 MiB without it."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("calls without operands: only where nothing can be launched")
    lib = _lib.load()
    for dtype, T, E, K, H, I in (("fp8", 48033, 8, 1, 512, 1024), ("bf16", 32465, 8, 1, 512, 1024), ("int8", 15449, 16, 2, 576, 1024)):
        t = traits(dtype).pod()
        a = _lib.FusedMoeArgs(num_tokens=T, num_experts=E, topk=K, hidden_size=H, intermediate_size=I)
        assert lib.mi355_fused_moe_static_ws(C.byref(t), C.byref(a), None) == _lib.E_HIP, lib.mi355_moe_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("case", FUSED, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}")
def test_fused_moe_of_far_rows(case):
    import torch
    import therock_amd as ta
    from therock_amd import inputs as mi
    from tests.gpu_reference import fused_moe_fp32
    dtype, fq, T, E, K, H, I, zipf = case
    print(f"far rows {case}", flush=True)
    cfg = mi.MoeConfig("far", T, H, I, E, K, dtype, "zipf" if zipf else "softmax_renorm")
    inp = mi.make_inputs_torch(cfg, "cuda", 7)
    t = traits(dtype, fq)
    x, scale, extra = inp["a"], inp["a_scale"], {}
    if fq == 1:  # (smooth scales of 1: every slot of a token holds its row)
        x, scale = x.repeat(K, 1), scale.repeat(K)
        extra["y_smooth_scale_ptr"] = torch.ones((E, I), dtype=torch.float32, device="cuda")

    def run(rows, out):
        buf = ta.MoeBuffers(t, T, E, K, H, I, "cuda")
        args = ta.make_args(t, buf, rows, inp["g"], inp["d"], inp["topk_ids"], inp["topk_weight"], a_scale=scale,
                            g_scale=inp["g_scale"], d_scale=inp["d_scale"])
        args.num_tokens, args.a_ptr, args.o_ptr = T, rows.data_ptr(), out.data_ptr()
        for k, v in extra.items():
            setattr(args, k, v)
        assert ta.fused_moe(t, args) == 0.0
        torch.cuda.synchronize()

    stride = pitch(dtype, x.shape[0])
    far_x = torch.empty((x.shape[0], stride), dtype=x.dtype, device="cuda")[:, :H]
    far_x.copy_(x)
    out = torch.empty((T, stride), dtype=torch.bfloat16, device="cuda")[:, :H]
    run(far_x, out)
    near = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    run(x, near)
    ref = fused_moe_fp32(cfg, inp)
    for got in (out, near):
        err = float((got.float() - ref).norm() / ref.norm())
        rows = (got.float() - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-30)
        print(f"  rel-L2 = {err:.3e}, worst row {float(rows.max()):.3e}", flush=True)
        # as in the oracle tests: 8-bit intermediate activations, or 16-bit ones
        assert err <= (1e-2 if dtype == "bf16" else 3e-2) and float(rows.max()) <= 1e-1


@pytest.mark.gpu
def test_stand_alone_down_gemm_of_far_rows():
    import torch
    import therock_amd as ta
    from tests.gpu_util import run_sorting
    T, E, K, I, H = 2500, 8, 4, 1728, 512
    stride = pitch("bf16", T * K)
    print("far rows: stand-alone int8 x bf16 down GEMM", flush=True)
    rng = np.random.default_rng(5)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(T)]).astype(np.int32)
    w = rng.random((T, K), dtype=np.float32)
    s_ids, s_w, s_eid, total = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in run_sorting(ids, w, E, 32, fill=True))
    gen = torch.Generator(device="cuda").manual_seed(3)
    far = torch.empty((T * K, stride), dtype=torch.bfloat16, device="cuda")
    y = far[:, :I]
    y.copy_(torch.randn((T * K, I), generator=gen, device="cuda"))
    d = torch.randint(-127, 128, (E, H, I), generator=gen, device="cuda", dtype=torch.int8)
    sd = torch.rand((E, H), generator=gen, device="cuda") * 1e-3 + 1e-3
    c = torch.zeros((T, H), dtype=torch.bfloat16, device="cuda")
    assert ta.moe_flatmm(ta.GEMM2, far, d, c, s_ids, s_eid, total.to(torch.int32), T, K, 32, sorted_weights=s_w, scale_n=sd) == 0.0
    torch.cuda.synchronize()
    near = torch.zeros_like(c)
    assert ta.moe_flatmm(ta.GEMM2, y.contiguous(), d, near, s_ids, s_eid, total.to(torch.int32), T, K, 32, sorted_weights=s_w, scale_n=sd) == 0.0
    torch.cuda.synchronize()
    ref = torch.zeros((T * K, H), device="cuda")
    e_of = torch.from_numpy(ids.reshape(-1)).cuda()
    for e in range(E):
        m = e_of == e
        ref[m] = (y[m].float() @ d[e].float().T) * sd[e]
    ref = (ref.reshape(T, K, H) * torch.from_numpy(w).cuda()[..., None]).sum(1)
    for got in (c, near):
        assert float((got.float() - ref).norm() / ref.norm()) <= 1e-2
