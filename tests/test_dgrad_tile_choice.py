"""Plain data gradients in bf16 without a tiling from the caller, on both sides of the reduction length from which 128 x 128 on eight
wavefronts may run beside weight gradients, by kernel name on the CPU."""
import pytest

import test_recorded_launches as R


@pytest.mark.parametrize("rows,cols,depth,eight", [
    (4096, 768, 2048, False), (4096, 768, 2112, True), (4096, 768, 50304, True), (3072, 768, 2304, True),
    (4096, 3072, 768, False), (18816, 256, 1024, False), (8192, 768, 768, False)])
def test_reduction_length(rows, cols, depth, eight):
    from sirius_amd._lib import check, lib
    rec = R.Recorder()
    try:
        rec.begin()
        check(lib().tch_conv2d_dgrad(rec.ctx, R.BF16, *[R.address(i) for i in range(3)], None, None, rows, 1, 1, cols, depth, 1, 1, 1, 0,
                                     -1, 0, 1))
        (name, _, _), = rec.end()
    finally:
        rec.close()
    assert name.startswith("igemm2_kernel<bf16,dgrad,") and ("128x128,3buf,8w" in name) == eight and "128x128,2buf,8w" not in name


@pytest.mark.parametrize("rows,cols,depth", [(8192, 3072, 768), (8192, 2304, 768), (25088, 512, 512)])
def test_large_grids_without_the_short_steps(rows, cols, depth):
    """TCH_IGEMM_K32=0 takes away the one tiling that the rules leave to such a grid: still no tile smaller than 128 x 128."""
    (name,) = R.in_own_process("""
rec.begin()
T.check(T.lib().tch_conv2d_dgrad(rec.ctx, T.BF16, a(0), a(1), a(2), None, None, %d, 1, 1, %d, %d, 1, 1, 1, 0, -1, 0, 1))
print(rec.end()[0][0], end="")
""" % (rows, cols, depth), TCH_IGEMM_K32="0")
    assert name.startswith("igemm2_kernel<bf16,dgrad,128x128,") and ",k32" not in name
