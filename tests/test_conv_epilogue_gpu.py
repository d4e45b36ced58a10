"""What a convolution's epilogue reads beside its accumulators (addend, scale and bias, the operands of the BatchNorm sums) is
requested ahead of its use, all at once or in groups: every tiling, at ragged edges, with the addend in place of the output and
with per-column vectors that are not 16-byte aligned."""
import pytest
import torch

import test_ops_gpu as T
from oracle import nn_ops as O

pytestmark = pytest.mark.gpu
TILES = [0, 1, 2, 3, 5, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, 24]
# one row, rows and columns beyond a tile's edge, a band more than a tile
CASES = [(1, 1, 1, 64, 8, 1, 1, 1, 0), (3, 7, 13, 64, 200, 1, 1, 1, 0), (1, 17, 17, 128, 136, 3, 3, 1, 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("tile_cfg", TILES)
def test_addend_in_place_and_unaligned_columns(ctx, dtype, case, tile_cfg):
    from sirius_amd import ops
    N, H, W, C, K, R, S, st, pad = case
    g = T._gen(41)
    x, w = T.rnd((N, H, W, C), dtype, g), T.rnd((K, R, S, C), dtype, g, (R * S * C) ** -0.5)
    add = T.rnd((N, H, W, K), dtype, g)
    scale, shift = torch.rand(K, generator=g) + 0.5, torch.randn(K, generator=g)
    off = lambda t: torch.cat([torch.zeros(1), t]).cuda()[1:]      # 4 bytes past a 16-byte boundary
    y = add.cuda()
    ops.conv2d_fwd_affine(ctx, x.cuda(), w.cuda(), y, st, pad, scale=off(scale), shift=off(shift), residual=y, tile_cfg=tile_cfg)
    torch.cuda.synchronize()
    T.close(y, O.conv2d_fwd(x, w, st, pad) * scale + shift + add.float(), dtype, "forward, addend in place")
    dy, dadd = T.rnd((N, H, W, K), dtype, g), T.rnd((N, H, W, C), dtype, g)
    dx = dadd.cuda()
    ops.conv2d_dgrad(ctx, dy.cuda(), ops.filter_transpose(ctx, w.cuda()), dx, st, pad, add=dx, tile_cfg=tile_cfg)
    torch.cuda.synchronize()
    T.close(dx, O.conv2d_dgrad(dy, w, (N, H, W, C), st, pad) + dadd.float(), dtype, "data gradient, addend in place")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tile_cfg", TILES)
def test_sums_with_a_compact_addend(ctx, dtype, tile_cfg):
    """All four operands at once: the addend on every second pixel, the BatchNorm's input and the ReLU's output."""
    from sirius_amd import ops
    N, H, W, C, K = 2, 13, 11, 136, 64
    g = T._gen(42)
    dy, w = T.rnd((N, H, W, K), dtype, g), T.rnd((K, 1, 1, C), dtype, g, K ** -0.5)
    sub, z, relu = T.rnd((N, 7, 6, C), dtype, g), T.rnd((N, H, W, C), dtype, g), T.rnd((N, H, W, C), dtype, g)
    mean, invstd = torch.randn(C, generator=g), torch.rand(C, generator=g) + 0.5
    ref = O.conv2d_dgrad(dy, w, (N, H, W, C), 1, 0)
    ref[:, ::2, ::2] += sub.float()
    ref = ref.to(dtype).float() * (relu.float() > 0)
    gx = torch.empty((N, H, W, C), dtype=dtype, device="cuda")
    partial = torch.full((ops.conv2d_dgrad_stat_rows(gx, K, 1, 1, 1, 0, tile_cfg) * C * 2,), float("nan"), device="cuda")
    ops.conv2d_dgrad_bnsums(ctx, dy.cuda(), ops.filter_transpose(ctx, w.cuda()), gx, 1, 0, z.cuda(), mean.cuda(), invstd.cuda(),
                            partial, bn_mask=relu.cuda(), add=sub.cuda(), add_stride=2, tile_cfg=tile_cfg)
    torch.cuda.synchronize()
    T.close(gx, ref, dtype, "gated gradient")
    sums = partial.cpu().view(-1, C, 2).double().sum(0)
    g64 = gx.double().cpu().view(-1, C)                           # the sums are those of what was stored
    xhat = (z.double().view(-1, C) - mean.double()) * invstd.double()
    T.close(sums[:, 0].float(), g64.sum(0).float(), torch.float32, "sum g", rtol=1e-4)
    T.close(sums[:, 1].float(), (g64 * xhat).sum(0).float(), torch.float32, "sum g*xhat", rtol=1e-4)
