"""Convolutions on the tilings with pipelined operand reads: the cases of the other tilings, and reductions around the
number of tiles in flight (1 to 6 steps: fewer than, as many as and more than the four tiles in LDS)."""
import pytest
import torch

import test_conv_split_gpu as P
import test_ops_gpu as T

pytestmark = pytest.mark.gpu
TILES = [21, 22]
STEPS = [(130, 1, 1, 64 * k, 200, 1, 1, 1, 0) for k in range(1, 7)]


@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", P.CASES + STEPS)
def test_forward_and_data_gradient(ctx, case, tile_cfg):
    T.test_conv_fwd(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad(ctx, torch.bfloat16, case, tile_cfg)


@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", P.CASES[:5])
def test_batchnorm_sums(ctx, case, tile_cfg):
    T.test_conv_with_bn_statistics(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad_with_bn_backward_sums(ctx, torch.bfloat16, case, tile_cfg, True)


@pytest.mark.parametrize("rows", [1, 70, 1000])
def test_order_of_additions_does_not_depend_on_the_rows(ctx, rows):
    """tile_cfg = IN_ORDER: the first rows of a product are the same bits at every number of rows."""
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randn(4100, 1, 1, 1536, device="cuda", generator=g).bfloat16()
    w = torch.randn(512, 1, 1, 1536, device="cuda", generator=g).bfloat16()
    outs = []
    for n in (rows, 4100):
        y = torch.empty(n, 1, 1, 512, dtype=torch.bfloat16, device="cuda")
        ops.conv2d_fwd(ctx, x[:n].contiguous(), w, y, 1, 0, tile_cfg=ops.IN_ORDER)
        outs.append(y[:rows])
    ctx.synchronize()
    assert torch.equal(outs[0], outs[1])
