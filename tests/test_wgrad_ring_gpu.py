"""bf16 weight gradients of 64 x 64 on both sides of the line between their two rings of LDS tiles (60 steps of 32 pixels per split),
and around the number of tiles in each: against the oracle, and the same bits whichever ring a split's steps take."""
import pytest
import torch

import test_ops_gpu as T
from oracle import nn_ops as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 4, 5, 6, 8, 9, 59, 60, 61, 64])
@pytest.mark.parametrize("geometry", [(1, 0), (3, 1)])
def test_steps(ctx, steps, geometry):
    from sirius_amd import ops
    R, pad = geometry
    W = 8
    H = (32 * steps - 24) // W + 1                       # the last step is ragged: 8 to 24 pixels short of whole
    g = T._gen(60 + steps)
    C, K = 72, 136
    x, dy = T.rnd((1, H, W, C), torch.bfloat16, g), T.rnd((1, H, W, K), torch.bfloat16, g)
    ref = O.conv2d_wgrad(x, dy, (K, R, R, C), 1, pad)
    dw, db = torch.full((K, R, R, C), 7.0, device="cuda"), torch.full((K,), 7.0, device="cuda")
    ops.conv2d_wgrad(ctx, x.cuda(), dy.cuda(), dw, 1, pad, splits=1, tile_cfg=2, dbias=db)
    torch.cuda.synchronize()
    T.close(dw, ref, torch.float32, "weight gradient", rtol=1e-3)
    T.close(db, dy.float().reshape(-1, K).sum(0), torch.float32, "bias gradient", rtol=1e-3)
    # one split of many steps and several of few: the same products, added up in another order
    sp = 4
    ws = torch.empty(ops.conv2d_wgrad_workspace_bytes(ops.dtype_code(x), K, R, R, C, sp) // 4 + 64, device="cuda")
    dw2 = torch.empty_like(dw)
    ops.conv2d_wgrad(ctx, x.cuda(), dy.cuda(), dw2, 1, pad, splits=sp, workspace=ws, tile_cfg=2)
    torch.cuda.synchronize()
    T.close(dw2, ref, torch.float32, "weight gradient, split", rtol=1e-3)
