"""Re-quantised intermediate rows of every length class (a wave, 256 or 512 threads, more than those hold): codes at their
boundaries, and rows with NaN in them, read back through down weights of the identity.  A gate-only layer whose every activation
is 64 (silu(64) in fp32); the smooth scale makes the values of it."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_quant_boundaries import boundary_rows, e4m3_codes


def codes_times_scale(v, dtype):
    import torch
    import therock_amd as ta
    T, inter = v.shape
    st, one = (torch.int8, 1) if dtype == "int8" else (torch.uint8, 0x38)
    view = torch.int8 if dtype == "int8" else torch.float8_e4m3fn
    H = 256  # the down weights bring the first 128 and the last 128 columns to the output
    a = torch.zeros((T, H), dtype=st, device="cuda")
    g = torch.zeros((T, inter, H), dtype=st, device="cuda")
    d = torch.zeros((T, H, inter), dtype=st, device="cuda")
    a[:, 0], g[:, :, 0] = one, one
    shown = torch.cat([torch.arange(128), torch.arange(inter - 128, inter)]).cuda()
    d[:, torch.arange(H, device="cuda"), shown] = one
    traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, gate_only=1, fused_quant=1)
    buf = ta.MoeBuffers(traits, T, T, 1, H, inter, "cuda")
    args = ta.make_args(traits, buf, a.view(view), g.view(view), d.view(view), torch.arange(T, dtype=torch.int32, device="cuda").reshape(T, 1),
                        torch.ones((T, 1), device="cuda"), a_scale=torch.full((T,), 64.0, device="cuda"),
                        g_scale=torch.ones(g.shape[:2], dtype=torch.float32, device="cuda"), d_scale=torch.ones((T, H), device="cuda"))
    args.y_smooth_scale_ptr = torch.from_numpy(v / 64).cuda().contiguous()
    assert ta.fused_moe(traits, args) == 0.0
    torch.cuda.synchronize()
    return buf.out.float().cpu().numpy(), shown.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["int8", "fp8"])
@pytest.mark.parametrize("inter", [1920, 2048, 2176, 6272, 8192, 8320, 12544, 16384, 16512])
def test_codes_of_rows_of_every_length(inter, dtype):
    import torch
    print(f"requantised rows {dtype} {inter}", flush=True)
    v = boundary_rows(dtype, [0, 0, -30, 40, 98, -101, 112], inter, inter)
    rng = np.random.default_rng(inter)
    nan = v[:2].copy()
    nan[0, rng.integers(0, 128, 20)] = np.nan
    nan[1, inter - 128:] = np.nan
    v = np.concatenate([v, nan, np.zeros((1, inter), np.float32)])
    got, shown = codes_times_scale(v, dtype)
    amax = np.nanmax(np.abs(v), axis=1, keepdims=True)
    scale = amax / np.float32(127 if dtype == "int8" else 448)
    q = (v / np.where(amax > 0, scale, np.float32(1)))[:, shown]
    # a NaN is code 0 in int8 and, clamped first, the least one in e4m3
    q = np.where(np.isnan(q), np.float32(0 if dtype == "int8" else -448), q)
    codes = np.rint(q) if dtype == "int8" else oracle.e4m3_to_f32(e4m3_codes(q))
    want = torch.from_numpy(codes.astype(np.float32) * scale).to(torch.bfloat16).float().numpy()
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["int8", "fp8"])
@pytest.mark.parametrize("inter", [256, 2176, 8320])  # a wave, 256 and 512 threads to a row
def test_rows_past_the_padded_list_are_left_alone(inter, dtype):
    """A row count larger than the padded list: the launch covers whole rounds of rows, and none past the list is touched, whatever
    the sorted ids after it say.  Output and workspace are those of a count that ends with the list's last unit."""
    import torch
    import therock_amd as ta
    T, E, H, unit, past = 5, 2, 128, 32, 4096
    view = torch.int8 if dtype == "int8" else torch.float8_e4m3fn
    traits = ta.fused_moe_traits(prec_i=dtype, prec_w=dtype, block_m=unit, gate_only=1, fused_quant=2)
    buf = ta.MoeBuffers(traits, T, E, 1, H, inter, "cuda")
    rows = -(-buf.max_pad // unit) * unit
    ids = np.full(256, (1 << 24) | T, np.int32)  # padding: slot topk of token `tokens`
    ids[:3], ids[unit:unit + 2], ids[rows:] = (0, 1, 2), (3, 4), 0
    assert buf.max_pad < rows < 128 <= len(ids)
    buf.sorted_ids = torch.from_numpy(ids).cuda()
    buf.sorted_w = torch.ones(len(ids), device="cuda")
    buf.sorted_eid = torch.tensor([0] + [1] * 7, dtype=torch.int32, device="cuda")
    gen = torch.Generator().manual_seed(inter)
    code = lambda *n: torch.randint(-60, 60, n, generator=gen).float().to(view).cuda()
    args = ta.make_args(traits, buf, code(T, H), code(E, inter, H), code(E, H, inter), torch.zeros((T, 1), dtype=torch.int32, device="cuda"),
                        torch.ones((T, 1), device="cuda"), a_scale=torch.full((T,), 0.01, device="cuda"),
                        g_scale=torch.full((E, inter), 0.01, device="cuda"), d_scale=torch.full((E, H), 0.01, device="cuda"))
    seen = []
    for total in (rows, past):
        print(f"rows past the list: {dtype} {inter}, count {total}", flush=True)
        buf.ws.fill_(0xA5)
        buf.total[0] = total
        assert ta.fused_moegemm(traits, args) == 0.0
        torch.cuda.synchronize()
        seen.append((buf.out.clone(), buf.ws.clone()))
    assert float(seen[0][0].float().abs().max()) > 0 and bool(torch.isfinite(seen[0][0].float()).all())
    assert torch.equal(seen[0][0], seen[1][0]) and torch.equal(seen[0][1], seen[1][1])
