"""The choice of the second lane's stream when a two-lane program is recorded."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def record(ctx, x, w, ys):
    from sirius_amd import ops
    prog = ops.Program()
    ctx.begin_record(prog)
    ops.conv2d_fwd(ctx, x, w, ys[0], 1, 0)
    with ctx.side_lane(wait_main=True):
        ops.conv2d_fwd(ctx, x, w, ys[1], 1, 0)
    ctx.join()
    ctx.end_record()
    return prog


@pytest.fixture
def operands():
    gen = torch.Generator(device="cuda").manual_seed(0)
    x, w = (torch.randn(n, 1, 1, 64, dtype=torch.bfloat16, device="cuda", generator=gen) for n in (32, 64))
    return x, w, [torch.zeros(32, 1, 1, 64, dtype=torch.bfloat16, device="cuda") for _ in range(2)]


@pytest.mark.parametrize("own_main", [False, True])
def test_second_lane_of_an_idle_chip_is_shown_to_run_beside_the_first(operands, own_main):
    from sirius_amd import ops
    kept = []
    for _ in range(6):
        ctx = ops.Context(torch.cuda.Stream() if own_main else torch.cuda.current_stream())
        assert ctx.second_lane() is None
        torch.cuda.synchronize()
        kept += [record(ctx, *operands), ctx, torch.cuda.Stream()]
        assert ctx.second_lane() is True
