"""The stand-alone down GEMM finds a slot's row through a map that nothing resets: whatever the workspace held before, slots
that the sorted list leaves out (experts of other ranks) must not get a row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,H,I,unit", [(5, 6, 3, 256, 128, 32), (70, 8, 2, 512, 1024, 32), (300, 4, 2, 256, 256, 64)])
@pytest.mark.parametrize("before", ["positions", "minus one", "large"])
def test_stale_map(T, E, K, H, I, unit, before):
    import torch
    import therock_amd as ta
    from tests.gpu_util import run_sorting

    rng = np.random.default_rng(T)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(T)]).astype(np.int32)
    w = rng.random((T, K), dtype=np.float32)
    mask = (np.arange(E) < E // 2).astype(np.int32)
    s_ids, s_w, s_eid, total = run_sorting(ids, w, E, unit, mask=mask)
    dev = lambda a: torch.from_numpy(a).cuda()
    y = torch.randn((T * K, I), generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).cuda()
    d = (torch.randn((E, H, I), generator=torch.Generator().manual_seed(2)) * 0.05).to(torch.bfloat16).cuda()
    a = (y, d, torch.zeros((T, H), dtype=torch.bfloat16, device="cuda"), dev(s_ids), dev(s_eid), dev(total.astype(np.int32)), T, K, unit)
    words = -(-ta.moe_flatmm_get_workspace_size(ta.GEMM2, *a) // 4)
    fill = {"positions": rng.integers(0, int(total[0]), words), "minus one": np.full(words, -1), "large": rng.integers(2 ** 30, 2 ** 31, words)}
    ws = dev(fill[before].astype(np.int32)).view(torch.uint8)
    print(f"stale map of {before}: {T} tokens", flush=True)
    assert ta.moe_flatmm(ta.GEMM2, *a, sorted_weights=dev(s_w), workspace=ws) == 0.0
    torch.cuda.synchronize()
    rows = y.float().cpu().reshape(T, K, I)
    df = d.float().cpu()
    want = torch.zeros((T, H))
    for t in range(T):
        for k in range(K):
            if mask[ids[t, k]]:
                want[t] += float(w[t, k]) * (df[ids[t, k]] @ rows[t, k])
    got = a[2].float().cpu()
    # rows and output rounded to bf16 (2^-9 each, relative)
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -8
