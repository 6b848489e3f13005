"""Quantisation of many short rows, a wave each: the same bytes as the workgroup form gives for the same rows called in small
batches (which the other tests compare with the oracle), around a lane's pieces and with a last workgroup that is not full."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("rows,cols", [(8, 8), (513, 512), (522, 520), (1027, 1024), (1033, 1032), (2050, 2048), (2055, 2040)])
def test_a_wave_gives_what_a_workgroup_gives(rows, cols, kind):
    import torch
    import therock_amd as ta
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + cols)
    x = torch.randn((rows, cols), generator=gen, device="cuda") * torch.exp2(torch.randint(-40, 40, (rows, 1), generator=gen, device="cuda").float())
    x[1] = 0
    x[2, :3] = torch.tensor([float("nan"), 1.0, -1.0], device="cuda")
    x[3, cols - 1] = float("inf")
    x = x.to(torch.bfloat16)
    E, K = 5, 3
    sm = torch.rand((E, cols), generator=gen, device="cuda") + 0.5
    ids = torch.randint(0, E, (rows, K), generator=gen, device="cuda", dtype=torch.int32)
    few = max(1, min(7, cols - 1))
    for first in (0, rows - few):
        part = slice(first, first + few)
        (q, s), (qp, sp) = ta.rowwise_quant(x, kind), ta.rowwise_quant(x[part].contiguous(), kind)
        torch.cuda.synchronize()
        assert torch.equal(q.view(torch.uint8)[part], qp.view(torch.uint8)) and torch.equal(s.view(torch.int32)[part], sp.view(torch.int32))
        (q, s), (qp, sp) = ta.moe_smoothquant(x, sm, ids, kind), ta.moe_smoothquant(x[part].contiguous(), sm, ids[part].contiguous(), kind)
        torch.cuda.synchronize()
        assert torch.equal(q.view(torch.uint8)[:, part], qp.view(torch.uint8)) and torch.equal(s.view(torch.int32)[:, part], sp.view(torch.int32))
