"""The work a user of this package has it do, as cases that can be timed and compared.

Every case is one call sequence through an engine: the training step the scripts under ``sirius_amd/train`` run for a
micro-batch (forward, loss, backward, optimizer; with gradient accumulation where a global batch is made of several
micro-batches), or the forward-only request the colocated inference tenant serves (``sirius_amd/serve.py``).

    listed()              the cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   engine, recorded plan and inputs, on the GPU
    run(state)            one pass; returns everything the pass computes
    work(case)            bytes and flops one pass cannot do without
    tolerance(case)       how far another correct implementation at the same precision may be off
"""
import math

import torch

from sirius_amd.gpt2 import GPT2Engine
from sirius_amd.resnet import ResNetEngine
from sirius_amd.swin import SwinEngine

IMAGE, CLASSES = 224, 1000
RESNET_DEPTHS, RESNET_WIDTH = (3, 8, 36, 3), 64                 # ResNet-152
SWIN_EMBED, SWIN_DEPTHS = 128, (2, 2, 18, 2)                    # Swin-B
GPT_VOCAB, GPT_WIDTH, GPT_LAYERS = 50257, 768, 12               # GPT-2 small


# ------------------------------------------------------------------------------------------------------- the cases
def _request(batch):
    return dict(model="resnet152", mode="request", batch=batch, dtype="bf16")


def _resnet(batch, dtype="bf16", micro=1):
    return dict(model="resnet152", mode="train", batch=batch, dtype=dtype, micro=micro)


def _swin(batch):
    return dict(model="swin_b", mode="train", batch=batch, dtype="bf16", micro=1)


def _gpt2(batch, seq, dtype="bf16", optimizer="adamw"):
    return dict(model="gpt2", mode="train", batch=batch, seq=seq, dtype=dtype, optimizer=optimizer, micro=1)


def listed():
    return [
        # one request of the colocated inference tenant: the smallest call, latency decides
        dict(_request(1), name="resnet152_request_1"),
        # requests gathered into a batch
        dict(_request(24), name="resnet152_request_24"),
        # the headline configuration: bench.py and the default micro-batch of train/resnet152.py
        dict(_resnet(64), name="resnet152_train_64"),
        # what a handover leaves of it (64 -> 16): two micro-batches accumulated into one global batch
        dict(_resnet(16, micro=2), name="resnet152_train_2x16"),
        # the ragged last micro-batch of a global batch of 500 cut into micro-batches of 32
        dict(_resnet(20), name="resnet152_train_20"),
        # the single-precision training step (train/resnet152.py --fp32)
        dict(_resnet(4, dtype="fp32"), name="resnet152_train_4_fp32"),
        # GPT-2 small at its full context: the most work of any step here
        dict(_gpt2(8, 1024), name="gpt2_train_8x1024"),
        # the defaults of train/gpt2.py: 8 sequences of 256 tokens, SGD
        dict(_gpt2(8, 256, optimizer="sgd"), name="gpt2_train_8x256_sgd"),
        # a context length nobody rounded to a tile, a micro-batch of a few sequences
        dict(_gpt2(3, 777), name="gpt2_train_3x777"),
        # train/gpt2.py --fp32 on the micro-batch a handover leaves
        dict(_gpt2(2, 256, dtype="fp32"), name="gpt2_train_2x256_fp32"),
        # the default micro-batch of train/swin_b.py
        dict(_swin(32), name="swin_b_train_32"),
        # a small, odd micro-batch of it
        dict(_swin(7), name="swin_b_train_7"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_any(rng):
    kind = rng.choice(("request",) * 3 + ("resnet",) * 4 + ("gpt2",) * 5 + ("swin",) * 3 + ("resnet_fp32",) + ("gpt2_fp32",) * 2)
    if kind == "request":
        return _request(_log_int(rng, 1, 64))
    if kind == "resnet":
        micro = rng.choice((1, 1, 2))
        return _resnet(_log_int(rng, 2, 64 if micro == 1 else 16), micro=micro)
    if kind == "swin":
        return _swin(_log_int(rng, 2, 32))
    if kind == "gpt2":      # any length, or one that is whole tiles of 128 tokens; at most the tokens of the largest listed case
        seq = rng.choice((_log_int(rng, 64, 1024), 128 * rng.randint(1, 8)))
        return _gpt2(_log_int(rng, 1, min(16, 8192 // seq if seq % 128 == 0 else max(1, 3072 // seq))), seq,
                     optimizer=rng.choice(("adamw", "sgd")))
    if kind == "resnet_fp32":
        return _resnet(rng.randint(1, 4), dtype="fp32")
    seq = _log_int(rng, 64, 512)
    return _gpt2(_log_int(rng, 1, max(1, 640 // seq)), seq, dtype="fp32")


def draw(rng):
    """One more case: micro-batches, sequence lengths, optimizers and types over the range the listed cases span."""
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw_any(rng)
        if case not in known:
            return case


# --------------------------------------------------------------------------------------- what a program has in hand
def _settle_resnet(eng):
    """The reference trains from pretrained weights; there is no checkpoint here, and fifty blocks of random ones with every
    BatchNorm gain at one are chaotic: a last-bit difference flips ReLU gates, and the gradients of two correct
    implementations have little in common.  Gains below one on the residual branches and shifts that keep most gates
    open leave a network whose gradients are a stable function of its inputs."""
    for name, p in eng.spec.items():
        if name.endswith("bn3.weight"):
            eng.params[p.offset:p.offset + p.numel].fill_(0.1)
        elif p.kind == "bn_b" and not name.endswith("bn3.bias"):
            eng.params[p.offset:p.offset + p.numel].fill_(3.0)
    eng.refresh_shadow()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    batch, dtype = case["batch"], torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    if case["model"] == "gpt2":
        eng = GPT2Engine(seq_len=case["seq"], dtype=dtype, optimizer=case["optimizer"], lr=1e-4)
        eng.init_normal(seed)
        inputs = [(torch.randint(0, GPT_VOCAB, (batch, case["seq"]), device="cuda", generator=gen),)]
    else:
        if case["model"] == "resnet152":
            eng = ResNetEngine(RESNET_DEPTHS, CLASSES, RESNET_WIDTH, dtype=dtype, image_size=IMAGE, lr=1e-3)
            eng.init_kaiming(seed)
            _settle_resnet(eng)
        else:
            eng = SwinEngine(dtype=dtype, lr=1e-4)
            eng.init_normal(seed)
        inputs = [(torch.randn(batch, 3, IMAGE, IMAGE, device="cuda", generator=gen),
                   torch.randint(0, CLASSES, (batch,), device="cuda", generator=gen)) for _ in range(case.get("micro", 1))]
    if case["mode"] == "request":
        eng.eval_plan(batch)                             # records the program of a request
    else:
        eng.plan(batch, 1.0 / case["micro"])             # records the program of a micro-batch
        if case["micro"] > 1:
            eng.ensure_global_grads()
    torch.cuda.synchronize()
    return dict(case=case, eng=eng, inputs=inputs)


def _sections(eng, flat):
    """A flat buffer of a transformer in pieces: what is outside its blocks, and every block or stage.  (Gradients of the
    first layers are tens of times the size of the others: in pieces each is compared with values of its own size.)"""
    starts, last = [], None
    for name, p in eng.spec.items():
        parts = name.split(".")
        key = ".".join(parts[:3]) if parts[1:2] == ["h"] else ".".join(parts[:2])
        if key != last:
            starts.append(p.offset)
            last = key
    return [flat[a:b] for a, b in zip(starts, starts[1:] + [flat.numel()])]


def run(state):
    case, eng, inputs = state["case"], state["eng"], state["inputs"]
    if case["mode"] == "request":
        return eng.forward_eval(inputs[0][0]).logits
    micro = case["micro"]
    for sample in inputs:
        plan, _ = eng.forward_backward(*sample, loss_scale=1.0 / micro)
        if micro > 1:
            eng.accumulate()
    eng.optimizer_step(use_global=micro > 1)
    out = dict(loss=plan.loss, logits=plan.logits, params=eng.params)
    if case["model"] == "resnet152":
        out.update(momentum=eng.momentum_buf, running_mean=eng.running_mean, running_var=eng.running_var)
        if micro == 1:                                   # accumulated gradients are zeroed by the step that takes them
            out.update(grads=eng.grads)
        return out
    flats = [eng.grads] + ([eng.momentum_buf] if case.get("optimizer") == "sgd" else [eng.exp_avg, eng.exp_avg_sq])
    cut = state.get("sections")
    if cut is None:
        cut = state["sections"] = [_sections(eng, f) for f in flats]
    out.update(state=cut)
    return out


# --------------------------------------------------------------------------------- what a pass cannot do without
def _resnet_layers():
    """(filter elements, output pixels, output channels) of every convolution, and of the classifier."""
    layers, side, cin = [(64 * 49 * 3, 112 * 112, 64)], 56, 64
    for i, depth in enumerate(RESNET_DEPTHS):
        p = RESNET_WIDTH << i
        for b in range(depth):
            out = side // (2 if i > 0 and b == 0 else 1)
            layers += [(cin * p, side * side, p), (9 * p * p, out * out, p), (4 * p * p, out * out, 4 * p)]
            if b == 0:
                layers.append((4 * p * cin, out * out, 4 * p))
            side, cin = out, 4 * p
    return layers + [(cin * CLASSES, 1, CLASSES)]


def work(case):
    """Flops of the matrix products.  Bytes: inputs, weights and optimizer state as the step reads and writes them, and for
    a training step what the forward pass has to leave for the backward pass, written once and read once."""
    eb, batch = (2 if case["dtype"] == "bf16" else 4), case["batch"]
    if case["model"] == "gpt2":
        rows, params, adam = batch * case["seq"], 124439808, case["optimizer"] == "adamw"
        product = 2.0 * rows * GPT_WIDTH * (12 * GPT_WIDTH * GPT_LAYERS + GPT_VOCAB)
        scores = 2.0 * rows * case["seq"] * GPT_WIDTH * GPT_LAYERS        # q k' and p v over the causal half
        saved = rows * (16 * GPT_WIDTH * GPT_LAYERS + GPT_VOCAB)
        return {"bytes": 2 * saved * eb + params * (28 if adam else 20), "flops": 3 * product + 3.5 * scores}
    images = batch * 3 * IMAGE * IMAGE * 4
    if case["model"] == "swin_b":
        saved, product, side, width = 0, 2.0 * (48 * SWIN_EMBED * 56 * 56 + 1000 * 1024), 56, SWIN_EMBED
        for i, depth in enumerate(SWIN_DEPTHS):
            tokens = side * side
            saved += depth * tokens * 16 * width
            product += depth * 2.0 * tokens * (12 * width * width + 2 * 49 * width)
            if i + 1 < len(SWIN_DEPTHS):
                product += 2.0 * tokens // 4 * 8 * width * width
                side, width = side // 2, 2 * width
        return {"bytes": images + 2 * saved * batch * eb + 87768224 * 28, "flops": 3 * product * batch}
    layers = _resnet_layers()
    weights, forward = sum(w for w, _, _ in layers), 2.0 * batch * sum(w * pixels for w, pixels, _ in layers)
    if case["mode"] == "request":
        return {"bytes": images + weights * eb + batch * CLASSES * 4, "flops": forward}
    micro = case["micro"]
    saved = batch * sum(pixels * channels for _, pixels, channels in layers)
    stem = 2.0 * batch * layers[0][0] * layers[0][1]                      # the input image gets no gradient
    state = weights * 20 + (weights * 12 * micro if micro > 1 else 0)     # SGD with momentum; accumulation
    return {"bytes": micro * (images + 2 * saved * eb) + state, "flops": micro * (3 * forward - stem)}


def tolerance(case):
    """A last-bit difference in one layer's bf16 activations is two to ten thousandths in the logits and about a hundredth
    in the gradients of the first layers, where single elements of small tensors are off by more; single precision
    keeps 1e-6 and loses two digits to ReLU gates that flip in fifty blocks."""
    if case["mode"] == "request":
        return {"rel": 1e-2}
    return {"rel": 2e-2, "max": 0.9} if case["dtype"] == "bf16" else {"rel": 1e-4, "max": 0.05}
