"""Swin's forward products in bf16 add every reduction up front to back, the classifier among them: no tiling that splits a
reduction over wavefronts is in the forward part of a plan, and an image's logits are the same bits in every batch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_forward_products_keep_one_order_and_logits_do_not_depend_on_the_batch():
    from sirius_amd.swin import SwinEngine
    eng = SwinEngine(dtype=torch.bfloat16, lr=1e-4)       # Swin-B: the classifier is 1024 -> 1000 over as many rows as images
    eng.init_normal(3)
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(40, 3, 224, 224, device="cuda", generator=gen)
    y = torch.randint(0, 1000, (40,), device="cuda", generator=gen)
    first = None
    for batch in (1, 7, 40):
        plan, _ = eng.forward_backward(x[:batch].contiguous(), y[:batch].contiguous())
        eng.ctx.synchronize()
        got = plan.logits.clone()
        names = [s["name"] for s in eng.ctx.profile_launches(plan.prog)[:plan.n_forward]]
        split = [n for n in names if n.startswith("igemm4")]
        assert any(n.startswith("igemm") for n in names) and not split, (batch, split)
        first = got[:1] if first is None else first
        assert torch.equal(got[:1], first), batch
        eng.release_activations()
