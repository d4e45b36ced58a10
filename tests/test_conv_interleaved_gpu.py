"""Convolutions on the interleaved tilings (128 x 128 with two and three tiles in LDS, 128 x 64, 128 x 192, 256 x 256): the cases
of the other tilings, reductions around the number of tiles in flight, and the bits of the plain loop."""
import pytest
import torch

import test_conv_split_gpu as P
import test_ops_gpu as T

gpu = pytest.mark.gpu
TILES = [0, 10, 22, 23, 24]
STEPS = [(130, 1, 1, 64 * k, 200, 1, 1, 1, 0) for k in range(1, 6)]     # up to three tiles in flight; 200 columns: a ragged tile
# the same for data gradients, whose reduction runs over K and the taps
DGRAD_STEPS = ([(130, 1, 1, 200, 64 * k, 1, 1, 1, 0) for k in range(1, 8)] +
               [(3, 9, 7, 136, 64, 3, 3, 1, 1), (2, 9, 11, 200, 128, 3, 3, 1, 1), (3, 9, 7, 136, 64, 3, 3, 2, 1), (2, 13, 10, 200, 192, 3, 3, 2, 1)])


@gpu
@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", P.CASES + STEPS)
def test_forward_and_data_gradient(ctx, case, tile_cfg):
    T.test_conv_fwd(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad(ctx, torch.bfloat16, case, tile_cfg)


@gpu
@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", DGRAD_STEPS)
def test_data_gradient_steps(ctx, case, tile_cfg):
    T.test_conv_dgrad(ctx, torch.bfloat16, case, tile_cfg)


@gpu
@pytest.mark.parametrize("tile_cfg", [23, 24])
@pytest.mark.parametrize("case", P.CASES[:5])
def test_batchnorm_sums(ctx, case, tile_cfg):
    T.test_conv_with_bn_statistics(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad_with_bn_backward_sums(ctx, torch.bfloat16, case, tile_cfg, True)


@gpu
@pytest.mark.parametrize("case", [(1000, 1, 1, 832, 520, 1, 1, 1, 0), (3, 15, 13, 128, 200, 3, 3, 1, 1), (2, 16, 16, 64, 392, 3, 3, 2, 1),
                                  (1000, 1, 1, 448, 320, 1, 1, 1, 0), (3, 15, 13, 320, 192, 3, 3, 1, 1), (2, 16, 16, 192, 448, 3, 3, 2, 1)])
def test_every_interleaved_tiling_adds_in_the_same_order(ctx, case):
    """Tiling 9 is the plain loop.  Forward in every case, the data gradient in those whose K is whole steps (another kernel runs
    in the others)."""
    from sirius_amd import ops
    N, H, W, C, K, R, S, st, pad = case
    g = T._gen(51)
    x, w = T.rnd((N, H, W, C), torch.bfloat16, g).cuda(), T.rnd((K, R, S, C), torch.bfloat16, g, 0.05).cuda()
    Ho, Wo = ops.conv_out_hw(H, W, R, S, st, pad)
    dy = T.rnd((N, Ho, Wo, K), torch.bfloat16, g).cuda()
    wt = ops.filter_transpose(ctx, w)
    want = None
    for tile_cfg in [9] + TILES:
        y, dx = torch.empty((N, Ho, Wo, K), dtype=torch.bfloat16, device="cuda"), torch.empty_like(x)
        ops.conv2d_fwd(ctx, x, w, y, st, pad, tile_cfg=tile_cfg)
        if K % 64 == 0:
            ops.conv2d_dgrad(ctx, dy, wt, dx, st, pad, tile_cfg=tile_cfg)
        torch.cuda.synchronize()
        want = want or (y, dx)
        assert torch.equal(y, want[0]), tile_cfg
        assert K % 64 or torch.equal(dx, want[1]), tile_cfg


@pytest.mark.parametrize("dtype", [0, 1], ids=["f32", "bf16"])
@pytest.mark.parametrize("tile_cfg", [23, 24])
def test_names_and_row_tiles(dtype, tile_cfg):
    """Which kernel a number runs, where it exists and where it does not, and the row tiles its statistics are sized by."""
    from sirius_amd._lib import check, lib
    import test_recorded_launches as R
    rec = R.Recorder()
    try:
        for C, K in ((128, 256), (24, 40)):
            shape = (2, 14, 14, C, K, 3, 3, 1, 1)
            rec.begin()
            check(lib().tch_conv2d_fwd_bnstats(rec.ctx, dtype, *[R.address(i) for i in range(3)], *shape, tile_cfg, 0, R.address(3)))
            check(lib().tch_conv2d_dgrad_bnsums(rec.ctx, dtype, *[R.address(i) for i in range(3)], None, None, *shape, tile_cfg, 0,
                                                *[R.address(i) for i in range(3, 8)], 1))
            rows = (lib().tch_conv2d_fwd_stat_rows(dtype, *shape, tile_cfg), lib().tch_conv2d_dgrad_stat_rows(dtype, *shape, tile_cfg))
            for (name, wgs, _), row_tiles, cols, depth in zip(rec.end(), rows, (K, C), (C, K)):
                direct = dtype == 1 and depth % 64 == 0
                bm, bn = (128, 192) if direct and tile_cfg == 24 else (128, 128)
                assert f",{bm}x{bn}" in name and name.startswith("igemm2_kernel") == direct and (",rot" in name) == direct
                assert row_tiles == -(-2 * 14 * 14 // bm) and wgs == row_tiles * -(-cols // bn)
    finally:
        rec.close()
