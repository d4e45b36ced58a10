"""The persistent kernel for linear layers (tilings 25 - 27): the same bits as the other front-to-back tilings, wherever its tiles, steps
and operands end; and what the library's choice makes of it."""
import pytest
import torch

import test_recorded_launches as R

# rows, columns, reduction: less than a tile, ragged edges on both sides, one step per tile, several tiles per workgroup (more than 256
# of the smallest), tiles in groups of rows (more than eight columns of them)
SHAPES = [(40, 72, 64), (128, 192, 64), (130, 200, 128), (257, 1544, 192), (777, 2304, 768), (5000, 2312, 64), (34000, 128, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize("tile_cfg", [25, 26, 27])
@pytest.mark.parametrize("rows,cols,depth", SHAPES)
def test_bits_of_the_other_tilings(rows, cols, depth, tile_cfg):
    from sirius_amd import ops
    ctx = ops.Context()
    g = torch.Generator(device="cuda").manual_seed(rows)
    rand = lambda *shape, dtype=torch.bfloat16: torch.randn(*shape, device="cuda", generator=g).to(dtype)  # noqa: E731
    x, w, add, bias = rand(rows, 1, 1, depth), rand(cols, 1, 1, depth), rand(rows, 1, 1, cols), rand(cols, dtype=torch.float32)
    for kw in ({}, {"bias": bias}, {"add": add}, {"bias": bias, "add": add}):
        want, got = torch.empty_like(add), torch.full_like(add, float("nan"))
        ops.conv2d_fwd(ctx, x, w, want, 1, 0, tile_cfg=2, **kw)
        ops.conv2d_fwd(ctx, x, w, got, 1, 0, tile_cfg=tile_cfg, **kw)
        assert torch.equal(got, want), kw
    for kw in ({}, {"add": add}):
        want, got = torch.empty_like(add), torch.full_like(add, float("nan"))
        ops.conv2d_dgrad(ctx, x, w, want, 1, 0, tile_cfg=2, **kw)
        ops.conv2d_dgrad(ctx, x, w, got, 1, 0, tile_cfg=tile_cfg, **kw)
        assert torch.equal(got, want), kw


@pytest.mark.gpu
@pytest.mark.parametrize("tile_cfg", [25, 26, 27])
def test_against_64_bits(tile_cfg):
    """One rounding to bf16, whose 8 bits put a value at most 2^-8 of its size off, of 320 additions that round by 2^-24 of a
    partial sum each, which the sum of |x w| bounds."""
    from sirius_amd import ops
    ctx = ops.Context()
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(700, 1, 1, 320, device="cuda", generator=g).bfloat16()
    w = torch.randn(520, 1, 1, 320, device="cuda", generator=g).bfloat16()
    y = torch.empty(700, 1, 1, 520, device="cuda", dtype=torch.bfloat16)
    ops.conv2d_fwd(ctx, x, w, y, 1, 0, tile_cfg=tile_cfg)
    want = x.view(700, 320).double() @ w.view(520, 320).double().t()
    size = x.view(700, 320).double().abs() @ w.view(520, 320).double().abs().t()
    assert ((y.view(700, 520).double() - want).abs() <= 2.0 ** -8 * want.abs() + 322 * 2.0 ** -24 * size).all()


def name_of(op, rows, cols, depth, tile_cfg, dtype=R.BF16, bias=True, out_f32=0):
    from sirius_amd._lib import check, lib
    rec = R.Recorder()
    try:
        rec.begin()
        a = [R.address(i) for i in range(4)]
        if op == "fwd":
            check(lib().tch_conv2d_fwd(rec.ctx, dtype, a[0], a[1], a[2], None, None, a[3] if bias else None, out_f32, rows, 1, 1, depth, cols,
                                       1, 1, 1, 0, tile_cfg, 0))
        else:
            check(lib().tch_conv2d_dgrad(rec.ctx, dtype, a[0], a[1], a[2], None, None, rows, 1, 1, cols, depth, 1, 1, 1, 0, tile_cfg, 0, 1))
        (name, wgs, _), = rec.end()
    finally:
        rec.close()
    return name, wgs


@pytest.mark.parametrize("op,rows,cols,depth,walks", [
    ("fwd", 8192, 2304, 768, True), ("fwd", 196, 3072, 1024, False), ("fwd", 8192, 2304, 736, False), ("dgrad", 8192, 3072, 768, True),
    ("dgrad", 2560, 3072, 768, True), ("dgrad", 2559, 3072, 768, False), ("dgrad", 4096, 768, 2304, True)])
def test_choice(op, rows, cols, depth, walks):
    for in_order, linear in ((-1, -3), (-2, -4)):
        name, wgs = name_of(op, rows, cols, depth, linear)
        assert name.startswith("igemm5_kernel<bf16," + op) == walks, name
        assert (wgs <= 256) if walks else name == name_of(op, rows, cols, depth, in_order)[0]
        assert not name_of(op, rows, cols, depth, in_order)[0].startswith("igemm5_kernel")


def test_what_it_does_not_take():
    """fp32 outputs, fp32 and ragged reductions: the same choice as without it, or the tiling of the same rows that was asked for."""
    assert name_of("fwd", 8192, 2304, 768, -4, out_f32=1)[0] == name_of("fwd", 8192, 2304, 768, -2, out_f32=1)[0]
    for asked, stand_in in ((-3, -1), (-4, -2), (25, 0), (26, 0), (27, 0)):
        assert name_of("fwd", 8192, 2304, 768, asked, dtype=R.F32)[0] == name_of("fwd", 8192, 2304, 768, stand_in, dtype=R.F32)[0]
    for asked, stand_in in ((25, 24), (26, 23), (27, 23)):
        assert name_of("fwd", 8192, 2304, 768, asked, out_f32=1)[0] == name_of("fwd", 8192, 2304, 768, stand_in, out_f32=1)[0]
