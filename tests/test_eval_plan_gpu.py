"""The program of a request follows the engine's options, also where they are set after a first request."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_options_set_after_a_request_take_effect():
    from sirius_amd.resnet import ResNetEngine
    eng = ResNetEngine((1, 2, 2, 1), 64, 64, dtype=torch.bfloat16, image_size=96)
    eng.init_kaiming(0)
    x = torch.randn(17, 3, 96, 96, device="cuda", generator=torch.Generator(device="cuda").manual_seed(9))

    def request(batch):
        p = eng.forward_eval(x[:batch].contiguous())
        eng.ctx.synchronize()
        return p, p.logits.clone(), [s["name"] for s in eng.ctx.profile_launches(p.prog)]

    fast, fast_logits, names = request(1)
    assert any(n.startswith("igemm4") for n in names)          # reductions split over wavefronts
    eng.eval_in_order = True
    ordered, logits, names = request(1)
    assert ordered is not fast and not any(n.startswith("igemm4") for n in names)
    assert torch.equal(logits, request(17)[1][:1])
    eng.fuse_eval_bn = False
    apart, apart_logits, names = request(1)
    assert any(n.startswith("bn_apply") for n in names) and torch.equal(apart_logits, request(17)[1][:1])
    eng.eval_in_order, eng.fuse_eval_bn = False, True
    again, again_logits, _ = request(1)
    assert again is fast and torch.equal(again_logits, fast_logits)
