"""Fused attention over sequence lengths that are no whole tiles, against the oracle's attention."""
import pytest
import torch

from oracle import seq_ops as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from sirius_amd import ops
    return ops.Context(torch.cuda.current_stream())


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,T", [(2, 2, 1), (1, 2, 31), (2, 1, 63), (1, 1, 65), (2, 2, 127), (1, 2, 129), (1, 1, 192), (2, 1, 777)])
def test_any_length(ctx, B, H, T, causal):
    from sirius_amd import ops
    C, scale, guard = H * 64, 0.125, 512
    g = torch.Generator()
    g.manual_seed(T + causal)
    qkv = torch.randn(B, T, 3 * C, generator=g).bfloat16()
    dout = torch.randn(B, T, C, generator=g).bfloat16()

    def heads(t):
        return t.reshape(B, T, H, 64).permute(0, 2, 1, 3).float()
    q, k, v = (heads(t) for t in qkv.split(C, -1))
    o_ref, lse_ref = S.attention(q, k, v, scale, causal)
    grads_ref = S.attention_bwd(q, k, v, heads(dout), scale, causal)
    # every output lies between guard elements that no kernel may touch
    flat = qkv.cuda().view(-1)
    o = torch.full((guard + B * T * C + guard,), 7.0, dtype=torch.bfloat16, device="cuda")
    grad = torch.full((guard + B * T * 3 * C + guard,), 7.0, dtype=torch.bfloat16, device="cuda")
    lse, delta = (torch.full((B * H * T + guard,), 7.0, device="cuda") for _ in range(2))
    oi, gi = o[guard:], grad[guard:]
    st, so = (3 * C, T * 3 * C), (C, T * C)
    ops.flash_attn_fwd(ctx, flat, flat[C:], flat[2 * C:], oi, lse, B, H, T, st, so, scale, causal, any_length=True)
    ops.flash_attn_bwd(ctx, flat, flat[C:], flat[2 * C:], oi, dout.cuda().view(-1), lse, delta, gi, gi[C:], gi[2 * C:], B, H, T,
                       st, so, scale, causal, any_length=True)
    ctx.synchronize()

    def close(got, ref, what):
        assert (got.float() - ref).abs().max() <= 2e-2 * ref.abs().max() + 1e-6, what
    close(heads(oi[:B * T * C].cpu()), o_ref, "context")
    assert torch.allclose(lse[:B * H * T].cpu().view(B, H, T), lse_ref, atol=4e-3)
    got = gi[:B * T * 3 * C].cpu().view(B, T, 3 * C)
    for name, a, b in zip(("dq", "dk", "dv"), got.split(C, -1), grads_ref):
        ref_max = max(float(r.abs().max()) for r in grads_ref)     # T = 1: dq and dk are zero up to rounding
        assert (heads(a) - b).abs().max() <= 2e-2 * ref_max, name
    for t, n in ((o, B * T * C), (grad, B * T * 3 * C)):
        assert torch.all(t[:guard] == 7) and torch.all(t[guard + n:] == 7)
    for t in (lse, delta):
        assert torch.all(t[B * H * T:] == 7)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,T", [(1, 2, 320), (1, 2, 321), (2, 3, 384), (1, 1, 449), (65, 4, 64), (44, 6, 128), (86, 1, 330)])
def test_walk_groups(ctx, B, H, T, causal):
    """Up to 256 workgroups two groups of wavefronts walk the tiles of dK and dV, from six tiles of 64 on: both sides of the line
    (one of seven tiles: a group has a last turn without one), whole and ragged lengths, more workgroups than compute units."""
    test_any_length(ctx, B, H, T, causal)
