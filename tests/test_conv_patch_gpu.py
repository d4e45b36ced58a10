"""The 3x3 patch kernel (tilings 5, 28 - 31): forward and data gradient with every epilogue's sums, for every width class of its
patch, one to several channel blocks, ragged rows and columns."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILINGS = {5: 128, 28: 128, 29: 64, 30: 64, 31: 128}
# images, rows, columns, channels in, channels out: patches of three, four and (64-row tiles) six loads, one channel block
# and four, rows and columns that do not fill a tile, more tiles than compute units
SHAPES = [(1, 7, 7, 64, 64), (3, 9, 7, 256, 200), (2, 5, 15, 128, 72), (2, 14, 14, 256, 128), (1, 20, 31, 192, 64), (2, 3, 40, 128, 64),
          (2, 5, 63, 64, 136), (24, 28, 28, 128, 128)]


def rel(a, b):
    return float((a.double() - b.double()).abs().max() / b.double().abs().max())


@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("n,h,w,c,k", SHAPES)
def test_against_fp32(n, h, w, c, k, tile_cfg):
    """bf16 rounds an output by 2^-8 of its size at most; sums over up to 2304 values in fp32 add less than that again for the
    ones that cancel.  Sums are those of the stored values."""
    from sirius_amd import ops
    ctx = ops.Context()
    g = torch.Generator(device="cuda").manual_seed(n * 1000 + w)
    rand = lambda *shape: torch.randn(*shape, device="cuda", generator=g).bfloat16()  # noqa: E731
    x, wt = rand(n, h, w, c), rand(k, 3, 3, c)
    y = torch.full((n, h, w, k), float("nan"), device="cuda", dtype=torch.bfloat16)
    rows = ops.conv2d_fwd_stat_rows(x, k, 3, 3, 1, 1, tile_cfg)
    assert rows == -(-n * h * w // TILINGS[tile_cfg])
    part = torch.full((rows * k * 2,), float("nan"), device="cuda")
    ops.conv2d_fwd_bnstats(ctx, x, wt, y, 1, 1, part, tile_cfg=tile_cfg)
    ref = torch.nn.functional.conv2d(x.float().permute(0, 3, 1, 2), wt.float().permute(0, 3, 1, 2), padding=1).permute(0, 2, 3, 1)
    assert rel(y, ref) < 2.0 ** -8 + 1e-4
    sums = part.view(rows, k, 2).double().sum(0)
    flat = y.double().view(-1, k)
    assert rel(sums[:, 1], flat.square().sum(0)) < 1e-5
    assert float((sums[:, 0] - flat.sum(0)).abs().max()) < 1e-5 * float(flat.abs().sum(0).max())
    again = torch.empty_like(y)
    ops.conv2d_fwd_bnstats(ctx, x, wt, again, 1, 1, part, tile_cfg=tile_cfg)
    assert torch.equal(again, y)

    if k % 64:
        return
    dy, filt, bn_x, relu = rand(n, h, w, k), rand(c, 3, 3, k), rand(n, h, w, c), rand(n, h, w, c)
    mean, invstd = torch.randn(c, device="cuda", generator=g), torch.rand(c, device="cuda", generator=g) + 0.5
    dx = torch.full((n, h, w, c), float("nan"), device="cuda", dtype=torch.bfloat16)
    rows = ops.conv2d_dgrad_stat_rows(dx, k, 3, 3, 1, 1, tile_cfg)
    part = torch.full((rows * c * 2,), float("nan"), device="cuda")
    ops.conv2d_dgrad_bnsums(ctx, dy, filt, dx, 1, 1, bn_x, mean, invstd, part, bn_mask=relu, tile_cfg=tile_cfg)
    ref = torch.nn.functional.conv_transpose2d(dy.float().permute(0, 3, 1, 2), filt.float().permute(3, 0, 1, 2), padding=1)
    ref = ref.permute(0, 2, 3, 1) * (relu > 0)
    assert rel(dx, ref) < 2.0 ** -8 + 1e-4
    sums, flat = part.view(rows, c, 2).double().sum(0), dx.double().view(-1, c)
    xhat = (bn_x.double().view(-1, c) - mean.double()) * invstd.double()
    assert float((sums[:, 0] - flat.sum(0)).abs().max()) < 1e-5 * float(flat.abs().sum(0).max())
    assert float((sums[:, 1] - (flat * xhat).sum(0)).abs().max()) < 1e-5 * float((flat * xhat).abs().sum(0).max())


def test_tilings_give_the_same_bits():
    from sirius_amd import ops
    ctx = ops.Context()
    g = torch.Generator(device="cuda").manual_seed(3)
    x, wt = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in [(3, 14, 14, 256), (200, 3, 3, 256)])
    out = []
    for cfg in TILINGS:
        out.append(torch.empty(3, 14, 14, 200, device="cuda", dtype=torch.bfloat16))
        ops.conv2d_fwd(ctx, x, wt, out[-1], 1, 1, tile_cfg=cfg)
    torch.cuda.synchronize()
    assert all(torch.equal(out[0], o) for o in out[1:])


@pytest.mark.parametrize("shape", [(64, 56, 56, 64, 64), (32, 28, 28, 128, 128)])
@pytest.mark.parametrize("tile_cfg", [5, 28, 29, 30, 31])
def test_first_filters_are_waited_for(tile_cfg, shape):
    """With nine filter tiles in LDS the first channel block has fewer loads in flight than the later ones: a count that takes
    the next patch's loads of a block before it for granted lets a step read its filter early.  Beside another stream's work."""
    from sirius_amd import ops
    n, h, w, c, k = shape
    beside = torch.cuda.Stream()
    ctx, other = ops.Context(torch.cuda.current_stream()), ops.Context(beside)
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    x, wt, ox, ody = rand(n, h, w, c), rand(k, 3, 3, c), rand(64, 14, 14, 256), rand(64, 14, 14, 1024)
    odw = torch.zeros(1024, 1, 1, 256, device="cuda")
    ref = torch.empty(n, h, w, k, device="cuda", dtype=torch.bfloat16)
    ops.conv2d_fwd(ctx, x, wt, ref, 1, 1, tile_cfg=5)
    torch.cuda.synchronize()
    for i in range(30):
        y = torch.full_like(ref, float("nan"))
        torch.cuda.synchronize()
        for _ in range(i % 3):
            ops.conv2d_wgrad(other, ox, ody, odw, 1, 0)
        ops.conv2d_fwd(ctx, x, wt, y, 1, 1, tile_cfg=tile_cfg)
        torch.cuda.synchronize()
        assert torch.equal(y, ref), i
