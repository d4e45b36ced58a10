"""bf16 weight gradients of 64 x 64 on both sides of the line between their two rings of LDS tiles (60 steps of 32 pixels per split, for
the few workgroups here), and around the number of tiles in each: against the oracle, and the same bits from both rings."""
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
    H = (32 * steps - 24) // W + 1                       # the last step is ragged: 16 pixels short of whole
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


@pytest.mark.parametrize("steps,short", [(1, 31), (4, 1), (5, 8), (6, 17), (33, 0), (59, 23), (60, 1), (60, 16)])
@pytest.mark.parametrize("geometry", [(1, 0), (3, 1)])
def test_both_rings_give_the_same_bits(ctx, geometry, steps, short):
    """The short ring's result, and the full ring's on the same pixels with zeros behind them up to more than 60 steps."""
    from sirius_amd import ops
    R, pad = geometry
    pixels, C, K = 32 * steps - short, 72, 136
    g = T._gen(90 + steps)
    x, dy = T.rnd((1, pixels, 1, C), torch.bfloat16, g), T.rnd((1, pixels, 1, K), torch.bfloat16, g)
    ref = O.conv2d_wgrad(x, dy, (K, R, R, C), 1, pad)
    got = []
    for rows in (pixels, 32 * 61 - 5, 32 * 64):
        xz, dyz = torch.zeros((1, rows, 1, C), dtype=torch.bfloat16, device="cuda"), torch.zeros((1, rows, 1, K), dtype=torch.bfloat16, device="cuda")
        xz[:, :pixels], dyz[:, :pixels] = x.cuda(), dy.cuda()
        dw, db = torch.full((K, R, R, C), 7.0, device="cuda"), torch.full((K,), 7.0, device="cuda")
        ops.conv2d_wgrad(ctx, xz, dyz, dw, 1, pad, splits=1, tile_cfg=2, dbias=db)
        torch.cuda.synchronize()
        got.append((dw, db))
    T.close(got[0][0], ref, torch.float32, "weight gradient", rtol=1e-3)
    for dw, db in got[1:]:
        assert torch.equal(dw, got[0][0]) and torch.equal(db, got[0][1])
