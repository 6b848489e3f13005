"""The GEMMs' work list (an expert's rows without the padding behind its last token) and the one-workgroup sort that
writes it, at the edges of row blocks, sort units, waves and the sort's capacity."""
import numpy as np
import pytest

import oracle
from therock_amd import inputs as mi
from tests.test_gpu_fused_moe import TOL, oracle_out
from tests.test_gpu_sorting import check as check_sorting

pytestmark = pytest.mark.gpu

COUNTS = [1, 31, 32, 33, 0, 63, 64, 65, 2]  # tokens of every expert


@pytest.mark.parametrize("dtype", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("unit", [16, 48, 64, 128])
def test_rows_per_expert_at_block_and_unit_edges(unit, dtype):
    from tests.gpu_util import rel_l2, run_fused_moe
    cfg = mi.MoeConfig("edges", sum(COUNTS), 256, 256, len(COUNTS), 1, dtype, "softmax_renorm", unit=unit)
    inp = mi.make_inputs_np(cfg, 1)
    ids = np.random.default_rng(2).permutation(np.repeat(np.arange(len(COUNTS)), COUNTS)).astype(np.int32)
    inp["topk_ids"] = ids[:, None]
    for kw in ({}, {"unfused": True}):
        got, _ = run_fused_moe(cfg, inp, **kw)
        ref, _ = oracle_out(cfg, inp, None, 1, 0)
        assert np.all(np.isfinite(oracle.bf16_to_f32(got)))
        assert rel_l2(oracle.bf16_to_f32(got), ref) <= TOL[dtype], (unit, dtype, kw)


@pytest.mark.parametrize("tokens,experts,topk", [(1, 1, 1), (63, 2, 1), (64, 65, 1), (1023, 63, 1), (341, 256, 3), (1025, 255, 1),
                                                 (4096, 256, 4), (16384, 3, 1), (16385, 3, 1), (4096, 257, 4)])
def test_one_workgroup_sort_at_its_edges(tokens, experts, topk):
    rng = np.random.default_rng(tokens + experts)
    ids = np.argsort(rng.random((tokens, experts)), axis=1)[:, :topk].astype(np.int32)
    check_sorting(ids, rng.random((tokens, topk), dtype=np.float32), experts, 32)
    if experts > 1:
        check_sorting(np.minimum(ids, 1) if topk == 1 else ids, rng.random((tokens, topk), dtype=np.float32), experts, 48,
                      mask=(np.arange(experts) % 2 == 0).astype(np.int32))


@pytest.mark.parametrize("dtype", ["bf16", "int8"])
@pytest.mark.parametrize("masked", [False, True])
def test_scan_pass_lists_experts_of_many_tiles(masked, dtype):
    # more entries than the one-workgroup sort takes: one expert of hundreds of tiles, empty and masked ones between and last
    from tests.gpu_util import rel_l2, run_fused_moe
    counts = [0, 12001, 0, 33, 4000, 1, 500, 0]
    cfg = mi.MoeConfig("many_tiles", sum(counts), 128, 128, len(counts), 1, dtype, "softmax_renorm", unit=32)
    assert cfg.tokens > 16384  # kOneShotMaxEntries
    inp = mi.make_inputs_np(cfg, 3)
    inp["topk_ids"] = np.random.default_rng(4).permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.int32)[:, None]
    mask = np.array([1, 1, 0, 1, 1, 1, 0, 1], np.int32) if masked else None
    if masked:  # weights of the local experts only
        for k in ("g", "d", "g_scale", "d_scale"):
            inp[k] = None if inp[k] is None else inp[k][:int(mask.sum())]
    got, _ = run_fused_moe(cfg, inp, mask=mask)
    ref, _ = oracle_out(cfg, inp, mask)
    assert rel_l2(oracle.bf16_to_f32(got), ref) <= TOL[dtype]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("tokens,experts,topk", [(10240, 8, 1), (10241, 8, 1), (5123, 256, 2), (8192, 60, 2)])
def test_both_sorts_of_the_fused_call(tokens, experts, topk, masked):
    # around the size from which the fused call sorts in three launches: the stand-alone sort, in one workgroup up to here, and
    # the GEMMs on its arrays give the same bits
    from tests.gpu_util import run_fused_moe
    cfg = mi.MoeConfig("sorts", tokens, 128, 128, experts, topk, "bf16", "softmax_renorm", unit=32)
    inp = mi.make_inputs_np(cfg, 5)
    mask = (np.arange(experts) % 3 != 1).astype(np.int32) if masked else None
    if masked:
        for k in ("g", "d"):
            inp[k] = inp[k][:int(mask.sum())]
    (fused, a), (apart, b) = run_fused_moe(cfg, inp, mask=mask), run_fused_moe(cfg, inp, mask=mask, unfused=True)
    n = int(a.total[0])
    assert n == int(b.total[0]) and n > 0
    for x, y, m in ((a.sorted_ids, b.sorted_ids, n), (a.sorted_w, b.sorted_w, n), (a.sorted_eid, b.sorted_eid, n // 32)):
        assert np.array_equal(x[:m].cpu().numpy(), y[:m].cpu().numpy())
    assert np.array_equal(fused, apart)
