"""Convolutions on the tilings with pipelined operand reads: the cases of the other tilings, and reductions around the
number of tiles in flight (1 to 6 steps: fewer than, as many as and more than the four tiles in LDS)."""
import pytest
import torch

import test_conv_split_gpu as P
import test_ops_gpu as T

pytestmark = pytest.mark.gpu
TILES = [21, 22]
STEPS = [(130, 1, 1, 64 * k, 200, 1, 1, 1, 0) for k in range(1, 7)]


@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", P.CASES + STEPS)
def test_forward_and_data_gradient(ctx, case, tile_cfg):
    T.test_conv_fwd(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad(ctx, torch.bfloat16, case, tile_cfg)


@pytest.mark.parametrize("tile_cfg", TILES)
@pytest.mark.parametrize("case", P.CASES[:5])
def test_batchnorm_sums(ctx, case, tile_cfg):
    T.test_conv_with_bn_statistics(ctx, torch.bfloat16, case, tile_cfg)
    T.test_conv_dgrad_with_bn_backward_sums(ctx, torch.bfloat16, case, tile_cfg, True)


@pytest.mark.parametrize("rows", [1, 70, 1000])
def test_order_of_additions_does_not_depend_on_the_rows(ctx, rows):
    """tile_cfg = IN_ORDER: the first rows of a product are the same bits at every number of rows."""
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randn(4100, 1, 1, 1536, device="cuda", generator=g).bfloat16()
    w = torch.randn(512, 1, 1, 1536, device="cuda", generator=g).bfloat16()
    outs = []
    for n in (rows, 4100):
        y = torch.empty(n, 1, 1, 512, dtype=torch.bfloat16, device="cuda")
        ops.conv2d_fwd(ctx, x[:n].contiguous(), w, y, 1, 0, tile_cfg=ops.IN_ORDER)
        outs.append(y[:rows])
    ctx.synchronize()
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layernorm_sums_that_ride_a_weight_gradient(ctx, dtype):
    """dgamma / dbeta from the next trailing weight gradient, from the backward behind it, and from the flush: the same
    bits as from the launch of their own."""
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    rows, C, K = 700, 264, 72
    x, dy = (torch.randn(rows, C, device="cuda", generator=g).to(dtype) for _ in range(2))
    gamma, mean, rstd = torch.ones(C, device="cuda"), torch.zeros(rows, device="cuda"), torch.ones(rows, device="cuda")
    wx, wdy = (torch.randn(rows, 1, 1, n, device="cuda", generator=g).to(dtype) for n in (C, K))
    n_partial = ops.layernorm_bwd_partial_rows(rows) * C * 2
    sp = ops.conv2d_wgrad_splits(wx, K, 1, 1, 1, 0)
    half = ops.conv2d_wgrad_workspace_bytes(ops.dtype_code(wx), K, 1, 1, C, sp) // 4 + 64
    trail = ops.TrailingWgrad(ctx, torch.empty(2 * half, device="cuda"), half)

    def backward(ride):
        out = [torch.full((C,), 7.0, device="cuda") for _ in range(2)]
        ops.layernorm_bwd(ctx, dy, x, torch.empty_like(x), gamma, mean, rstd, *out, torch.empty(n_partial, device="cuda"), ride=ride)
        return out
    want = backward(False)
    dw, ref = torch.empty(K, 1, 1, C, device="cuda"), torch.empty(K, 1, 1, C, device="cuda")
    ops.conv2d_wgrad(ctx, wx, wdy, ref, 1, 0, workspace=torch.empty(half, device="cuda"), splits=sp)
    got = [backward(True), backward(True)]      # the first goes out with the second backward
    trail.wgrad(wx, wdy, dw, 1, 0)
    got.append(backward(True))
    trail.flush()
    ctx.synchronize()
    assert torch.equal(dw, ref)
    for pair in got:
        assert torch.equal(pair[0], want[0]) and torch.equal(pair[1], want[1])


def test_an_eager_reduction_does_not_enter_a_recording(ctx):
    """A reduction that pends when a recording begins is launched then; the program holds its own alone."""
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    rows, C, K = 2000, 72, 136
    x, dy = (torch.randn(rows, 1, 1, n, device="cuda", generator=g).bfloat16() for n in (C, K))
    sp = ops.conv2d_wgrad_splits(x, K, 1, 1, 1, 0)
    assert sp > 1
    half = ops.conv2d_wgrad_workspace_bytes(ops.dtype_code(x), K, 1, 1, C, sp) // 4
    trail = ops.TrailingWgrad(ctx, torch.empty(2 * half, device="cuda"), half)
    ref, eager, recorded = (torch.full((K, 1, 1, C), 7.0, device="cuda") for _ in range(3))
    ops.conv2d_wgrad(ctx, x, dy, ref, 1, 0, workspace=torch.empty(half, device="cuda"), splits=sp)
    trail.wgrad(x, dy, eager, 1, 0)
    prog = ops.Program()
    ctx.begin_record(prog)
    trail.wgrad(x, dy, recorded, 1, 0)
    ctx.end_record()
    ctx.synchronize()
    assert torch.equal(eager, ref) and (recorded == 7).all()
    eager.fill_(7)
    for _ in range(2):
        recorded.fill_(7)
        ctx.run(prog)
        ctx.synchronize()
        assert torch.equal(recorded, ref) and (eager == 7).all()
