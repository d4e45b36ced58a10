"""Tiling 32 (16 x 16 with the reduction over eight wavefronts) at the edges of its tiles and rings, against the CPU oracle: the
operator tests of test_ops_gpu.py run on it."""
import pytest
import torch

import test_ops_gpu as T

pytestmark = pytest.mark.gpu

CASES = [
    # N, H, W, C, K, R, S, stride, pad
    (1, 7, 7, 64, 64, 1, 1, 1, 0),        # fewer reduction steps than wavefronts, rows off the tile
    (1, 7, 9, 192, 72, 3, 3, 1, 1),       # a step count that is no multiple of the wavefronts, ragged columns
    (3, 14, 14, 64, 32, 3, 3, 2, 1),      # strided: taps that exist for every second pixel only
    (17, 1, 1, 1088, 200, 1, 1, 1, 0),    # one row over a tile, a deep pointwise reduction
    (1, 14, 14, 256, 256, 3, 3, 1, 1),    # nine steps a wavefront
    (1, 5, 5, 24, 40, 3, 3, 1, 1),        # channels that are no whole step: another kernel runs
]
dtypes = pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])   # fp32: tiling 16 runs


@pytest.fixture(scope="module")
def ctx():
    from sirius_amd import ops
    return ops.Context(torch.cuda.current_stream())


@dtypes
@pytest.mark.parametrize("case", CASES)
def test_forward_and_data_gradient(ctx, dtype, case):
    T.test_conv_fwd(ctx, dtype, case, 32)
    T.test_conv_dgrad(ctx, dtype, case, 32)


@dtypes
@pytest.mark.parametrize("case", CASES)
def test_batchnorm_sums(ctx, dtype, case):
    T.test_conv_with_bn_statistics(ctx, dtype, case, 32)
    T.test_conv_dgrad_with_bn_backward_sums(ctx, dtype, case, 32, True)


def test_statistics_keep_row_tiles_of_32():
    """Callers size the sums of a forward product for the row tiles of tiling 15, the smallest that the choice made for one."""
    from sirius_amd import ops
    for n, h, c, k, r in [(1, 14, 1024, 256, 1), (1, 14, 256, 256, 3), (1, 7, 512, 512, 3), (2, 7, 2048, 512, 1)]:
        x = torch.empty(n, h, h, c, dtype=torch.bfloat16, device="meta")
        assert ops.conv2d_fwd_stat_rows(x, k, r, r, 1, r // 2) <= ops.conv2d_fwd_stat_rows(x, k, r, r, 1, r // 2, 15)
