"""fp32 products in bf16 parts: as accurate as fp32, on every kernel that takes them, and with infinities, NaN and values next
to the largest one what fp32 makes of them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILINGS = [-1, 0, 1, 2, 15, 16, 17, 18, 19, 20]
# The second is multiplied in parts by every kernel that can (the first by none): ragged for every tile, more than 256 tiles of
# 128 x 128, eight reduction steps and a remainder for each of eight wavefronts.
SIZES = [(68, 72, 272), (2100, 2084, 1040)]
sizes = pytest.mark.parametrize("rows,cols,depth", SIZES)


def product(op, rows, cols, depth, tile_cfg, a, b):
    """a [rows, depth] times b [cols, depth] transposed, through the forward convolution, the data or the weight gradient"""
    from sirius_amd import ops
    ctx = ops.Context()
    if op == "fwd":
        y = torch.empty(rows, 1, 1, cols, device="cuda")
        ops.conv2d_fwd(ctx, a.view(rows, 1, 1, depth), b.view(cols, 1, 1, depth), y, 1, 0, tile_cfg=tile_cfg)
    elif op == "dgrad":
        y = torch.empty(rows, 1, 1, cols, device="cuda")
        ops.conv2d_dgrad(ctx, a.view(rows, 1, 1, depth), b.view(cols, 1, 1, depth), y, 1, 0, tile_cfg=tile_cfg)
    else:
        y = torch.empty(rows, 1, 1, cols, device="cuda")
        ops.conv2d_wgrad(ctx, b.t().contiguous().view(depth, 1, 1, cols), a.t().contiguous().view(depth, 1, 1, rows), y, 1, 0, splits=1,
                         tile_cfg=tile_cfg)
    torch.cuda.synchronize()
    return y.view(rows, cols)


def against_64_bits(op, rows, cols, depth, tile_cfg, a, b):
    """the product, what it is in 64 bits, and the sum of the sizes of its terms"""
    a64, b64 = a.double(), b.double()
    return product(op, rows, cols, depth, tile_cfg, a, b).double(), a64 @ b64.t(), a64.abs() @ b64.abs().t()


# depths on both sides of the line, with and without a remainder for the steps, the wavefronts and the LDS tiles
CASES = [(op, rows, cols, depth) for op in ("fwd", "dgrad", "wgrad")
         for rows, cols, depth in ((36, 40, 128), (36, 40, 144), (132, 200, 272), (64, 64, 1024), (260, 132, 656), (2100, 2084, 272), (2100, 2084, 1040))]


@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("op,rows,cols,depth", CASES)
def test_error_is_that_of_fp32(op, rows, cols, depth, tile_cfg):
    """Per value: every one of at most `depth` additions rounds by 2^-24 of a partial sum, which the sum of |a b| bounds, the
    parts leave out at most 2^-30 of every product and their own sum is 2^-5 as large."""
    g = torch.Generator().manual_seed(depth + rows)
    a = torch.randn(rows, depth, generator=g).mul_(torch.exp(2 * torch.randn(rows, depth, generator=g)))
    b = torch.randn(cols, depth, generator=g)
    got, want, size = against_64_bits(op, rows, cols, depth, tile_cfg, a.cuda(), b.cuda())
    assert ((got - want).abs() <= (depth + 2) * 2.0 ** -24 * size).all()
    # and over the whole result what sums of independent roundings have, not what the bound above allows
    assert (got - want).norm() <= 4 * 2.0 ** -24 * max(1, depth / 64) ** 0.5 * want.norm()


def fp32_multiplies(a, b, groups):
    """What v_mfma_f32_32x32x2_f32 gives: one rounding to fp32 per reduction element, steps of 16 elements dealt out to `groups`
    wavefronts, whose sums are added in their order.  (With fp64 inside: a product of two fp32 values is exact there.)"""
    total, a, b = None, a.double(), b.double()
    for group in range(groups):
        acc = torch.zeros(a.shape[0], b.shape[0], device=a.device)
        for k in range(a.shape[1]):
            if k // 16 % groups == group:
                acc = torch.addr(acc.double(), a[:, k], b[:, k]).float()
        total = acc if total is None else total + acc
    return total


# a value's distribution over a row; "wide": a few products of a sum dominate it, and its error is that of single products
DISTRIBUTIONS = {
    "normal": lambda shape, g: torch.randn(shape, device="cuda", generator=g),
    "relu": lambda shape, g: torch.randn(shape, device="cuda", generator=g).clamp_(min=0),
    "uniform": lambda shape, g: torch.rand(shape, device="cuda", generator=g),
    "wide": lambda shape, g: torch.randn(shape, device="cuda", generator=g) * torch.exp(3 * torch.randn(shape, device="cuda", generator=g)),
    "tiny": lambda shape, g: torch.randn(shape, device="cuda", generator=g) * 2.0 ** -118,
    "large": lambda shape, g: torch.randn(shape, device="cuda", generator=g) * 2.0 ** 80,
}
# tiling: wavefronts that share the reduction of a forward product or data gradient.  2 multiplies in fp32 there.
GROUPS = {0: 1, 1: 1, 2: 1, 15: 4, 16: 8, 17: 4, 18: 8, 19: 4, 20: 8}
PAIRS = [("normal", "normal"), ("relu", "normal"), ("uniform", "uniform"), ("wide", "normal"), ("wide", "wide"), ("tiny", "normal"), ("normal", "tiny"),
         ("tiny", "large")]


@sizes
@pytest.mark.parametrize("first,second", PAIRS)
def test_error_is_no_larger_than_with_fp32_multiplies(first, second, rows, cols, depth):
    """Against 64 bits, over a whole result, next to fp32 multiplies in the same order; every value counts by the sum of |a b|.  What is
    left out of a product and what the small products' sum rounds is 2^-5 of a unit in the last place where one product is all of a
    sum (test_single_products_are_rounded_once), against a rounding of 0.29 units: 0.6 % more; elsewhere parts round less often.
    The allowance of 3 % is that and what two sets of 4896 roundings differ by (2 %)."""
    g = torch.Generator("cuda").manual_seed(depth)
    a, b = DISTRIBUTIONS[first]((rows, depth), g), DISTRIBUTIONS[second]((cols, depth), g)
    want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    error = lambda y: ((y.double() - want) / size).norm().item()
    off = {groups: error(fp32_multiplies(a, b, groups)) for groups in (1, 4, 8)}
    for op in ("fwd", "dgrad", "wgrad"):
        for tile_cfg in (0, 2) if op == "wgrad" else GROUPS:
            groups = 1 if op == "wgrad" else GROUPS[tile_cfg]
            ratio = error(product(op, rows, cols, depth, tile_cfg, a, b)) / off[groups]
            print(f"{first} x {second} over {depth}, {op} tiling {tile_cfg}: {ratio:.3f}")
            assert ratio <= 1.03, (op, tile_cfg, ratio)
            if tile_cfg == 2 and op != "wgrad":   # fp32 multiplies: the reference is what they give
                assert ratio >= 0.97, (op, ratio)


@sizes
@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("op", ["fwd", "dgrad", "wgrad"])
def test_single_products_are_rounded_once(op, tile_cfg, rows, cols, depth):
    """Sums of one product and zeros: half a unit in the last place, as a product in fp32, and 2^-5 of a unit.  With both values in
    [1, 2) the second parts are below 2^-7 and the third below 2^-15: x2 y2, which is left out, is below 2^-30; the small products' sum
    is below 2^-5, so that each of the three additions that can round there does by 2^-30 at most.  A unit is at least 2^-23."""
    g = torch.Generator("cuda").manual_seed(4)
    a, b = torch.zeros(rows, depth, device="cuda"), torch.randn(cols, depth, device="cuda", generator=g)
    a[torch.arange(rows), torch.arange(rows) % depth] = torch.randn(rows, device="cuda", generator=g)
    got, want, _ = against_64_bits(op, rows, cols, depth, tile_cfg, a, b)
    unit = torch.exp2(torch.floor(torch.log2(want.abs())) - 23)
    assert ((got - want).abs() <= (0.5 + 2.0 ** -5) * unit).all()


@sizes
@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("op", ["fwd", "dgrad", "wgrad"])
@pytest.mark.parametrize("first,second", [(-112, 0), (0, -112), (-126, 100), (-70, -40), (-60, -60), (104, 0), (50, 50)])
def test_values_of_any_size_keep_their_bits(first, second, op, tile_cfg, rows, cols, depth):
    """Operands and results down to the smallest normal values and beyond what the parts hold: the bound of
    test_error_is_that_of_fp32, and for results the grid of the denormals, 2^-149, that the additions of a denormal sum round to."""
    g = torch.Generator().manual_seed(-first)
    a = (1 + torch.rand(rows, depth, generator=g)) * 2.0 ** first
    b = (1 + torch.rand(cols, depth, generator=g)) * 2.0 ** second * (1 - 2 * torch.randint(0, 2, (cols, depth), generator=g))
    got, want, size = against_64_bits(op, rows, cols, depth, tile_cfg, a.cuda(), b.cuda())
    assert ((got - want).abs() <= (depth + 2) * 2.0 ** -24 * size + depth * 2.0 ** -150).all()


@sizes
@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("op", ["fwd", "dgrad", "wgrad"])
def test_infinities_nan_and_the_largest_values(op, tile_cfg, rows, cols, depth):
    g = torch.Generator().manual_seed(1)
    a, b = torch.randn(rows, depth, generator=g), torch.randn(cols, depth, generator=g)
    inf, largest = float("inf"), torch.finfo(torch.float32).max
    a[3, 17], a[9, 200], a[33, 5], a[40, 271] = inf, float("nan"), largest, -largest
    a[50, 3], a[50, 100] = inf, -inf
    b[20, 17], b[21, 5], b[:, 271] = 0.0, 0.5, b[:, 271].clamp(-0.9, 0.9)
    a, b = a.cuda(), b.cuda()
    got, want, _ = against_64_bits(op, rows, cols, depth, tile_cfg, a, b)
    want = torch.where(want.abs() > largest, torch.sign(want) * inf, want)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    ok = want.isfinite()
    size = (torch.where(a.isfinite(), a, 0).double().abs() @ b.double().abs().t())[ok]
    assert ((got - want)[ok].abs() <= (depth + 2) * 2.0 ** -24 * size).all()


@sizes
@pytest.mark.parametrize("tile_cfg", TILINGS)
@pytest.mark.parametrize("op", ["fwd", "dgrad", "wgrad"])
def test_results_next_to_the_largest_value_are_finite(op, tile_cfg, rows, cols, depth):
    """The first part of a value may be larger than the value.  Products of first parts, and sums of such products, overflow then
    where the result does not: 1.999 * 2^127, and 253 times 1.0040^2 * 2^120 (0.996 * 2^128; 1.0078^2 in first parts)."""
    g = torch.Generator().manual_seed(2)
    a, b = torch.randn(rows, depth, generator=g), torch.randn(cols, depth, generator=g)
    for row, col, sign in ((5, 7, 1.0), (40, 50, -1.0)):
        a[row, 17], b[col, 17] = sign * 1.999 * 2.0 ** 63, 2.0 ** 64
    for row, col, sign in ((9, 11, 1.0), (66, 70, -1.0)):
        a[row, :253], b[col, :253] = sign * 1.0040 * 2.0 ** 62, 1.0040 * 2.0 ** 58
        a[row, 17] = b[col, 17] = 0.0     # leaves the others' large values alone
        a[row, 253], b[col, 253] = a[row, 0], b[col, 0]
    got, want, size = against_64_bits(op, rows, cols, depth, tile_cfg, a.cuda(), b.cuda())
    assert want.abs().max() < torch.finfo(torch.float32).max and (want.abs() > 2.0 ** 127).sum() >= 4
    assert ((got - want).abs() <= (depth + 2) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("op", ["fwd", "dgrad"])
def test_in_order_rows_are_the_same_bits_at_every_number_of_rows(op):
    """tile_cfg = IN_ORDER: 64 x 64 tiles, which multiply in fp32 anyway, up to 384 tiles of 128 x 64; those; and 128 x 128."""
    from sirius_amd import ops
    cols, depth = 128, 272
    g = torch.Generator("cuda").manual_seed(3)
    a, b = (torch.randn(n, depth, device="cuda", generator=g) for n in (49280, cols))
    first, *others = [product(op, rows, cols, depth, ops.IN_ORDER, a[:rows], b)[:66] for rows in (66, 24700, 49280)]
    assert all(torch.equal(first, o) for o in others)


@pytest.mark.parametrize("stride", [1, 2])
def test_convolutions_in_parts(stride):
    """3x3 layers with ragged edges on more than 256 tiles, where taps leave the image, the weight gradient with its reduction split,
    added to what is there and with the bias gradient.  Per value as in test_error_is_that_of_fp32."""
    from sirius_amd import ops
    ctx = ops.Context()
    g = torch.Generator("cuda").manual_seed(stride)
    n, side, c, k = 17 * stride * stride, 45, 80, 112
    out = ops.conv_out_hw(side, side, 3, 3, stride, 1)[0]
    x, w, dy = (torch.randn(*shape, device="cuda", generator=g) for shape in ((n, side, side, c), (k, 3, 3, c), (n, out, out, k)))

    def in_64_bits(x, w, dy):
        x = x.double().permute(0, 3, 1, 2).requires_grad_(True)
        w = w.double().permute(0, 3, 1, 2).requires_grad_(True)
        y = torch.nn.functional.unfold(x, 3, padding=1, stride=stride).transpose(1, 2).reshape(-1, 9 * c) @ w.reshape(k, -1).t()
        dx, dw = torch.autograd.grad(y, (x, w), dy.double().reshape(-1, k))
        return y.detach().view(dy.shape), dx.permute(0, 2, 3, 1), dw.permute(0, 2, 3, 1)

    want, size = in_64_bits(x, w, dy), in_64_bits(x.abs(), w.abs(), dy.abs())
    near = lambda got, i, depth: bool(((got.double() - want[i]).abs() <= (depth + 2) * 2.0 ** -24 * size[i]).all())
    y, dx = torch.empty_like(dy), torch.empty_like(x)
    for tile_cfg in (0, 1, 16, 17, 18, 19, 20):
        y.fill_(float("nan"))
        ops.conv2d_fwd(ctx, x, w, y, stride, 1, tile_cfg=tile_cfg)
        assert near(y, 0, 9 * c), tile_cfg
    for tile_cfg in (0, 1, 18, 19):
        dx.fill_(float("nan"))
        ops.conv2d_dgrad(ctx, dy, w.permute(3, 1, 2, 0).contiguous(), dx, stride, 1, tile_cfg=tile_cfg)
        assert near(dx, 1, 9 * k), tile_cfg
    pixels, splits = n * out * out, 60
    workspace = torch.empty(ops.conv2d_wgrad_workspace_bytes(0, k, 3, 3, c, splits) // 4, device="cuda")
    for tile_cfg in (0, 1, 2):
        dw, dbias = torch.ones_like(w), torch.ones(k, device="cuda")
        ops.conv2d_wgrad(ctx, x, dy, dw, stride, 1, workspace=workspace, splits=splits, accumulate=True, tile_cfg=tile_cfg, dbias=dbias)
        assert near(dw.double() - 1, 2, pixels), tile_cfg
        sums, sizes = dy.double().sum((0, 1, 2)), dy.double().abs().sum((0, 1, 2))
        assert ((dbias.double() - 1 - sums).abs() <= pixels * 2.0 ** -24 * sizes).all()
