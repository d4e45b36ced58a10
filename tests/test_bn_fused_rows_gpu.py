"""BatchNorm finalize + apply in one launch (bn_fin_apply_kernel): rows that end inside a trip, a slab or a pair of rows, and row
blocks around one trip of its sums (8 lanes x 8 row blocks), against the same arithmetic in double precision."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,C,blocks", [(9, 64, 1), (31, 64, 8), (33, 128, 9), (65, 64, 63), (1000, 256, 64), (4097, 64, 65),
                                           (8192 * 2 + 1, 64, 129), (12544, 1024, 256)])
def test_forward_and_backward(ctx, dtype, rows, C, blocks):
    from sirius_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + C)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, res, dy = (rnd(rows, C).to(dtype) for _ in range(3))
    gamma, beta = rnd(C) * 0.3 + 1, rnd(C)
    xd = x.double()
    blocks = min(blocks, rows)
    cuts = [rows * i // blocks for i in range(blocks + 1)]

    def sums(a, b):      # [blocks, C, 2], as a convolution's epilogue leaves them
        return torch.stack([torch.stack((a[i:j].sum(0), b[i:j].sum(0)), 1) for i, j in zip(cuts, cuts[1:])]).float().contiguous()
    part = sums(xd, xd * xd)
    rm, rv, sm, si = torch.zeros(C, device="cuda"), torch.ones(C, device="cuda"), *(torch.empty(C, device="cuda") for _ in range(2))
    y, scratch = torch.empty_like(x), torch.empty(3 * C, device="cuda")
    ops.bn_fwd_train_partials(ctx, x, y, gamma, beta, rm, rv, sm, si, part, blocks, scratch, residual=res, relu=True)
    mean, var = xd.mean(0), xd.var(0, unbiased=False)
    inv = 1 / torch.sqrt(var + 1e-5)
    ref = ((xd - mean) * inv * gamma.double() + beta.double() + res.double()).clamp_min(0)
    # one rounding of the result and of the coefficients.  The batch statistics come from sums rounded to fp32: their variance is
    # off by 2^-24 (mean^2 + var) / var, which is unbounded for a channel of two rows and below 1e-6 from nine rows of N(0, 1) on
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    ctx.synchronize()
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    assert rel(y, ref) < tol and rel(sm, mean) < 1e-5 and rel(si, inv) < 1e-5
    assert rel(rv, 0.9 + 0.1 * var * rows / (rows - 1)) < 1e-5
    dd, xhat = dy.double(), (xd - sm.double()) * si.double()
    part = sums(dd, dd * xhat)
    dx, dg, db = torch.empty_like(x), torch.zeros(C, device="cuda"), torch.zeros(C, device="cuda")
    ops.bn_bwd_partials(ctx, dy, x, dx, gamma, sm, si, dg, db, part, blocks, scratch)
    ctx.synchronize()
    ref = gamma.double() * si.double() * (dd - dd.mean(0) - xhat * (dd * xhat).mean(0))
    assert rel(dx, ref) < tol and rel(db, dd.sum(0)) < 1e-5 and rel(dg, (dd * xhat).sum(0)) < 1e-5
