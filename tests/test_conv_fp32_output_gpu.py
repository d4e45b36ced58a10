"""bf16 products stored in fp32 (an output head): the same sums as stored in bf16, every column once, nothing beyond the rows."""
import pytest
import torch

import test_ops_gpu as T

gpu = pytest.mark.gpu
GUARD = 4096


@gpu
@pytest.mark.parametrize("tile_cfg", [0, 1, 2, 9, 10, 12, 16, 21, 22, 23, 24])
@pytest.mark.parametrize("rows,cols", [(1, 8), (257, 264), (130, 200), (300, 1000)])
def test_fp32_output(ctx, rows, cols, tile_cfg):
    from sirius_amd import ops
    g = T._gen(61)
    x, w = T.rnd((rows, 1, 1, 128), torch.bfloat16, g).cuda(), T.rnd((cols, 1, 1, 128), torch.bfloat16, g, 0.05).cuda()
    bias = T.rnd((cols,), torch.float32, g).cuda()
    narrow = torch.empty((rows, 1, 1, cols), dtype=torch.bfloat16, device="cuda")
    ops.conv2d_fwd(ctx, x, w, narrow, 1, 0, tile_cfg=tile_cfg)
    outs = []
    for b in (None, bias):
        room = torch.full((rows * cols + 2 * GUARD,), float("nan"), device="cuda")
        y = room[GUARD:GUARD + rows * cols].view(rows, 1, 1, cols)
        ops.conv2d_fwd(ctx, x, w, y, 1, 0, tile_cfg=tile_cfg, bias=b)
        torch.cuda.synchronize()
        assert bool(room[:GUARD].isnan().all()) and bool(room[GUARD + rows * cols:].isnan().all())
        outs.append(y)
    assert torch.equal(outs[0].bfloat16(), narrow)               # one rounding of the same sums
    assert torch.equal(outs[1], outs[0] + bias)                  # the general route: one fp32 addition more
    want = x.view(rows, 128).double() @ w.view(cols, 128).double().t()
    # 128 products, exact in fp32, summed in fp32: at most 128 roundings of the largest partial sum
    bound = 128 * 2.0 ** -24 * (x.view(rows, 128).double().abs() @ w.view(cols, 128).double().abs().t())
    assert bool(((outs[0].view(rows, cols).double() - want).abs() <= bound).all())
