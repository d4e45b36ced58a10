"""The tile of a weight gradient without a tiling from the caller, on both sides of its line, by kernel name on the CPU."""
import pytest

import test_recorded_launches as R


@pytest.mark.parametrize("dtype,K,C,splits,side", [
    (R.F32, 128, 128 * 1023, 1, 64), (R.F32, 128, 128 * 1024, 1, 128), (R.F32, 4096, 4096, 1, 128), (R.F32, 768, 3072, 1, 64),
    (R.F32, 1024, 1024, 15, 64), (R.F32, 1024, 1024, 16, 128), (R.F32, 124, 128 * 2048, 1, 64),
    (R.BF16, 128, 128 * 127, 1, 64), (R.BF16, 128, 128 * 128, 1, 128), (R.BF16, 768, 3072, 1, 128)])
def test_tile(dtype, K, C, splits, side):
    from sirius_amd._lib import check, lib
    rec = R.Recorder()
    try:
        rec.begin()
        check(lib().tch_conv2d_wgrad(rec.ctx, dtype, *[R.address(i) for i in range(4)], splits, 0, 64 * splits, 1, 1, C, K, 1, 1, 1, 0, -1, 0))
        name, wgs, _ = rec.end()[0]
    finally:
        rec.close()
    assert f",{side}x{side}>" in name and wgs == -(-K // side) * -(-C // side) * splits
