"""The convolution tilings that split the reduction over the wavefronts of a workgroup (15 - 20), at the edges of their
tiles and rings, against the CPU oracle: the operator tests of test_ops_gpu.py run on them."""
import pytest
import torch

import test_ops_gpu as T
import test_recorded_launches as R

pytestmark = pytest.mark.gpu

CASES = [
    # N, H, W, C, K, R, S, stride, pad
    (1, 7, 7, 64, 64, 1, 1, 1, 0),        # fewer reduction steps than wavefronts (bf16: 2), rows and columns off the tile
    (1, 7, 9, 192, 72, 3, 3, 1, 1),       # a step count that is no multiple of the wavefronts, ragged columns
    (3, 14, 14, 64, 32, 3, 3, 2, 1),      # strided: taps that exist for every second pixel only
    (2, 16, 16, 64, 128, 1, 1, 2, 0),     # strided 1x1
    (65, 1, 1, 1088, 200, 1, 1, 1, 0),    # one row over a tile, a deep pointwise reduction
    (1, 5, 5, 24, 40, 3, 3, 1, 1),        # channels that are no whole step: another kernel runs
]
TILES = [15, 16, 17, 18, 19, 20]
dtypes = pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])


@dtypes
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("tile_cfg", TILES)
def test_forward_and_data_gradient(ctx, dtype, case, tile_cfg):
    T.test_conv_fwd(ctx, dtype, case, tile_cfg)
    T.test_conv_dgrad(ctx, dtype, case, tile_cfg)


@dtypes
@pytest.mark.parametrize("case", CASES[:5])
@pytest.mark.parametrize("tile_cfg", TILES)
def test_batchnorm_sums(ctx, dtype, case, tile_cfg):
    T.test_conv_with_bn_statistics(ctx, dtype, case, tile_cfg)
    T.test_conv_dgrad_with_bn_backward_sums(ctx, dtype, case, tile_cfg, True)


@dtypes
@pytest.mark.parametrize("rows,K,C", [(196, 256, 1024), (196, 512, 2048), (784, 512, 2048), (1024, 256, 1024), (4704, 256, 1024),
                                      (343, 1024, 1024), (2048, 768, 768)])
def test_library_choice(ctx, dtype, rows, K, C):
    """Products of few output tiles, on the library's own choice."""
    T.test_conv_fwd(ctx, dtype, (rows, 1, 1, C, K, 1, 1, 1, 0), -1)


@pytest.mark.parametrize("rows,K,C,want", R.F32_CHOICE)
def test_fp32_choice_on_both_sides_of_its_lines(ctx, rows, K, C, want):
    """`want` is what runs (held on the CPU by test_recorded_launches.py); here its results, forward and data gradient."""
    T.test_conv_fwd(ctx, torch.float32, (rows, 1, 1, C, K, 1, 1, 1, 0), -1)
    T.test_conv_dgrad(ctx, torch.float32, (rows, 1, 1, K, C, 1, 1, 1, 0), -1)


@dtypes
@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("splits", [1, 3])
def test_weight_gradient_ignores_the_split_tilings(ctx, dtype, tile_cfg, splits):
    """15 - 20 are no tilings of a weight gradient: the bits of tiling 2 (the same kernel), alone and with a pending
    reduction to take along, and both against the float64 product."""
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    rows, C, K = 500, 72, 136
    x, dy = (torch.randn(rows, 1, 1, n, device="cuda", generator=g).to(dtype) for n in (C, K))
    half = ops.conv2d_wgrad_workspace_bytes(ops.dtype_code(x), K, 1, 1, C, 8) // 4
    ws = torch.empty(2 * half, device="cuda")
    got, ref, other = (torch.empty(K, 1, 1, C, device="cuda") for _ in range(3))
    ops.conv2d_wgrad(ctx, x, dy, ref, 1, 0, workspace=ws, splits=splits, tile_cfg=2)
    ops.conv2d_wgrad(ctx, x, dy, got, 1, 0, workspace=ws, splits=splits, tile_cfg=tile_cfg)
    ctx.synchronize()
    want = (dy.double().view(rows, K).t() @ x.double().view(rows, C)).view_as(ref)
    # products of exact operands summed in fp32 over 500 rows: 500 * 2^-24 of the sum of magnitudes at the very worst
    scale = (dy.double().abs().view(rows, K).t() @ x.double().abs().view(rows, C)).view_as(ref)
    assert ((ref - want).abs() <= 500 * 2.0 ** -24 * scale).all()
    assert torch.equal(got, ref)
    trail = ops.TrailingWgrad(ctx, ws, half)
    trail.wgrad(x, dy, other, 1, 0)
    trail.wgrad(x, dy, got, 1, 0, tile_cfg=tile_cfg)
    trail.flush()
    ops.conv2d_wgrad(ctx, x, dy, ref, 1, 0, workspace=ws, splits=ops.conv2d_wgrad_splits(x, K, 1, 1, 1, 0), tile_cfg=2)
    ctx.synchronize()
    assert torch.equal(other, got) and torch.equal(got, ref)
