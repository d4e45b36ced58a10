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


def test_a_recording_leaves_another_threads_capture_alone(operands):
    """A graph is captured in global mode while the recording of a two-lane program ends in another thread, for the first time
    (a stream is made and asked about) and again: the graph is whole, replays right, and the program runs right."""
    import threading

    from sirius_amd import ops
    x, w, ys = operands
    a, b = torch.zeros(4096, device="cuda"), torch.zeros(4096, device="cuda")
    graph = torch.cuda.CUDAGraph()
    got, errors = [], []
    mains = [torch.cuda.Stream() for _ in range(2)]

    def other():
        try:
            for main in mains:
                ctx = ops.Context(main)
                got.append((ctx, record(ctx, x, w, ys)))
        except Exception as e:      # noqa: BLE001  (told to the main thread)
            errors.append(e)

    torch.cuda.synchronize()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        torch.mul(a, 2.0, out=b)
        t = threading.Thread(target=other)
        t.start()
        t.join()
        b.add_(1.0)
    assert not errors, errors
    for i in range(3):
        a.fill_(float(i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(b, torch.full_like(b, 2 * i + 1.0))
    want = (x.view(32, 64).float() @ w.view(64, 64).float().t())
    for ctx, prog in got:
        assert ctx.second_lane() is True
        for y in ys:
            y.zero_()
        torch.cuda.synchronize()
        ctx.run(prog)
        ctx.synchronize()
        for y in ys:
            assert (y.view(32, 64).float() - want).abs().max() <= 1e-2 * want.abs().max()
