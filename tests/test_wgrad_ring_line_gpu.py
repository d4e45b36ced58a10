"""bf16 weight gradients of 64 x 64 on both sides of the lines between their two rings of LDS tiles: compute units left free, one
workgroup on each, more than one; 32 to 61 steps of 32 pixels.  Against the product in float32."""
import pytest
import torch

import test_ops_gpu as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [32, 33, 60, 61])
@pytest.mark.parametrize("K,C", [(1024, 768), (1024, 776), (1024, 1024), (1024, 1032)])     # 192, 208, 256, 272 workgroups
def test_line(ctx, K, C, steps):
    from sirius_amd import ops
    rows = 32 * steps - 8
    g = T._gen(steps + C)
    x, dy = T.rnd((rows, 1, 1, C), torch.bfloat16, g), T.rnd((rows, 1, 1, K), torch.bfloat16, g)
    dw = torch.full((K, 1, 1, C), 7.0, device="cuda")
    ops.conv2d_wgrad(ctx, x.cuda(), dy.cuda(), dw, 1, 0, splits=1, tile_cfg=2)
    torch.cuda.synchronize()
    T.close(dw, (dy.view(rows, K).float().t() @ x.view(rows, C).float()).view(K, 1, 1, C), torch.float32, "weight gradient", rtol=1e-3)
