"""The workloads the framework's speed is measured on: what a training step of a compressed model has it do.

A case is one forward and backward pass of an operator module (or a compress / decompress round trip through
`kernels`, or one whole decoder layer) in its steady state: the module has made its calibration calls, as it has from
the third step of a run on.  `listed()` holds sizes of this repository's configurations (hidden 4096, intermediate
11008, batch 4 x 1024 or 1 x 2048) with a very short and a ragged batch beside them; `draw()` gives others of the same
ranges.  Data: N(0, 1) activations with 1 % of the channels x 20 as outliers, upstream gradients N(0, 0.02).
"""
import importlib
import math

import torch

hyc = importlib.import_module("hyc-lora_amd")
layers = importlib.import_module("hyc-lora_amd.decoder_layer")
K, ops = hyc.kernels, hyc.operators
BF16 = torch.bfloat16


# ---- the cases --------------------------------------------------------------------------------------------------
def listed():
    return [
        # the two halves of every saved activation by themselves: [4, 512, 4096], INT4 in groups of 128
        dict(name="round_trip", op="round_trip", tokens=2048, width=4096, bits=4, group=128),
        # one short sample: the smallest call there is, launches and host work are all of it
        dict(name="rmsnorm_short", op="rmsnorm", batch=1, seq=45, width=4096, bits=4, group=128, mode="hyc"),
        # the norm in front of attention and MLP at a long-context training batch
        dict(name="rmsnorm_train", op="rmsnorm", batch=8, seq=2048, width=4096, bits=4, group=128, mode="hyc"),
        # the reference's own scheme as its GSM8K preset sets it: rank 2, 8 bits per channel, outlier elements
        dict(name="rmsnorm_ref", op="rmsnorm", batch=4, seq=1024, width=4096, bits=8, group=128, mode="ref"),
        # encoder fine-tuning (GLUE): ragged batches of short sentences, narrow rows, weight and bias
        dict(name="layernorm_ragged", op="layernorm", batch=31, seq=117, width=1024, bits=8, group=128, mode="hyc"),
        # LoRA-A: [16, 4096] from an INT2 input, the weight gradient that every LoRA step computes seven times a layer
        dict(name="lora_a", op="linear", batch=4, seq=1024, width=4096, out=16, bits=2, group=64, mode="hyc"),
        # a linear layer that trains its whole weight from the same input
        dict(name="full_linear", op="linear", batch=4, seq=1024, width=4096, out=4096, bits=2, group=64, mode="hyc"),
        # act(gate) * up of the MLP with its three saved activations
        dict(name="gated_silu", op="gated", batch=4, seq=1024, width=11008, bits=4, group=128, mode="hyc"),
        # attention probabilities of 32 heads over 2048 positions, 1 % kept
        dict(name="softmax", op="softmax", batch=1, heads=32, seq=2048),
        # one short sample through a whole layer
        dict(name="layer_short", op="layer", batch=1, seq=157, hidden=2048, heads=16, inner=5632, rank=16, bits=8, attention="flash"),
        # a whole layer: NF4 base, LoRA on all seven projections, the reference's attention wiring
        dict(name="layer_eager", op="layer", batch=1, seq=2048, hidden=4096, heads=32, inner=11008, rank=16, bits=4, attention="eager"),
        # the same with fused attention, four sequences
        dict(name="layer_flash", op="layer", batch=4, seq=1024, hidden=4096, heads=32, inner=11008, rank=16, bits=4, attention="flash"),
    ]


def _between(rng, lo, hi):
    """a whole number, evenly spread over the logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["round_trip", "rmsnorm", "layernorm", "act", "linear", "gated", "softmax", "layer", "layer"])
    if op == "softmax":
        seq = 8 * _between(rng, 8, 256)
        return dict(op=op, batch=1, heads=max(1, min(64, _between(rng, 8, 1 << 27) // (seq * seq))), seq=seq)
    if op == "layer":
        hidden, heads, inner = rng.choice([(1024, 8, 2816), (2048, 16, 5632), (2048, 32, 5632), (4096, 32, 11008)])
        attention = rng.choice(["eager", "flash", "flash"])
        seq = _between(rng, 64 if hidden < 4096 else 512, 2048)
        if attention == "eager":
            seq = -(-seq // 32) * 32
        return dict(op=op, batch=rng.randint(1, max(1, min(8, 4096 // seq))), seq=seq, hidden=hidden, heads=heads, inner=inner,
                    rank=rng.choice([8, 16, 32]), bits=4 if inner > 8192 else 8, attention=attention)
    width = rng.choice([768, 1024, 1536, 2048, 3072, 4096, 5120, 8192, 11008, 13824])
    bits, group = rng.choice([(2, 64), (4, 64), (4, 128), (4, 128), (8, 128)])
    if op == "gated":
        width = max(width, 2048)
        bits = min(bits, 4)
    if width * bits // 8 % group:                       # a scale group lies within one segment of a packed row
        bits, group = 4, 64
    tokens = _between(rng, 16, min(65536, (1 << 27) // width))
    if op == "round_trip":
        return dict(op=op, tokens=tokens, width=width, bits=bits, group=group)
    batch = rng.randint(1, max(1, min(32, tokens // 16)))
    case = dict(op=op, batch=batch, seq=max(1, tokens // batch), width=width, bits=bits, group=group, mode="hyc")
    if op == "gated":
        case["seq"] = max(1, min(case["seq"], (1 << 26) // (width * batch)))
    if op == "linear":
        case["out"] = rng.choice([8, 16, 16, 32, 64, 256, 1024, 4096])
        case["seq"] = max(1, min(case["seq"], 8192 // batch if case["out"] > 64 else 65536 // batch))
    if op == "act":
        case["op"] = rng.choice(["silu", "gelu"])
    if op in ("rmsnorm", "layernorm", "act") and rng.random() < 0.3:
        case.update(mode="ref", bits=rng.choice([4, 8]))
        case["seq"] = min(case["seq"], 16384 // batch)
    return case


# ---- what a program has in hand -----------------------------------------------------------------------------------
def _activation(gen, shape, width, gain=20.0, outliers=0.01):
    x = torch.randn(shape + (width,), generator=gen, device="cuda")
    hot = torch.randperm(width, generator=gen, device="cuda")[:K.num_outlier_channels(width, outliers)]
    x[..., hot] *= gain
    return x.to(BF16)


def _gradient(gen, shape, std=0.02):
    return (std * torch.randn(shape, generator=gen, device="cuda")).to(BF16)


def _module(case):
    op, ref = case["op"], case.get("mode") == "ref"
    if op == "softmax":
        return ops.EfficientMemorySoftmax(outlier_ratio=0.01)
    how = dict(outlier_ratio=0.005 if ref else 0.01, sub_outlier_ratio=1.0, sub_outlier_bit=case["bits"],
               sub_outlier_quantize_method="per-channel", rank=2 if ref else 0)
    if op == "gated":
        return ops.EfficientMemoryGatedAct("silu", group_size=case["group"], **how)
    how.update(mode=case["mode"], group_size=case["group"])
    if op == "rmsnorm":
        return ops.EfficientMemoryRMSNorm(case["width"], eps=1e-6, bias=False, **how)
    if op == "layernorm":
        return ops.EfficientMemoryLayerNorm(case["width"], **how)
    if op == "linear":
        return ops.EfficientMemoryLinear(case["width"], case["out"], **how)
    return {"silu": ops.EfficientMemorySiLU, "gelu": ops.EfficientMemoryGELU}[op](**how)


def prepare(case, seed):
    torch.manual_seed(seed)                            # the reference scheme's rank-2 base comes from a random projection
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]
    if op == "round_trip":
        x = _activation(gen, (case["tokens"],), case["width"])
        plan = K.select_channels(K.channel_absmax(x), K.num_outlier_channels(case["width"], 0.01))
        return dict(op=op, x=x, plan=plan, bits=case["bits"], group=case["group"])
    if op == "layer":
        mod = layers.DecoderLayer(layers.LayerConfig(
            hidden=case["hidden"], heads=case["heads"], head_dim=case["hidden"] // case["heads"], intermediate=case["inner"],
            lora_r=case["rank"], lora_alpha=2.0 * case["rank"], linear_bits=8, act_bits=case["bits"], attention=case["attention"]))
        shape = (case["batch"], case["seq"])
        inputs = [_activation(gen, shape, case["hidden"])]
        g = _gradient(gen, shape + (case["hidden"],))
    elif op == "softmax":
        shape = (case["batch"], case["heads"], case["seq"], case["seq"])
        mod, inputs = _module(case), [(2 * torch.randn(shape, generator=gen, device="cuda")).to(BF16)]
        g = _gradient(gen, shape)
    else:
        mod, shape = _module(case).cuda().to(BF16), (case["batch"], case["seq"])
        with torch.no_grad():
            for name, p in mod.named_parameters():
                std = 0.02 if op == "linear" else 0.1
                p.copy_((op in ("rmsnorm", "layernorm") and name == "weight") + std * torch.randn(p.shape, generator=gen, device="cuda"))
        inputs = [_activation(gen, shape, case["width"]) for _ in range(2 if op == "gated" else 1)]
        g = _gradient(gen, shape + (case.get("out", case["width"]),))
    with torch.no_grad():
        for _ in range(2):                             # the calibration calls of a module's first two steps
            mod(*inputs)
    inputs = [t.requires_grad_(True) for t in inputs]
    return dict(op=op, mod=mod, inputs=inputs, wanted=inputs + list(mod.parameters()), g=g)


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(state):
    if state["op"] == "round_trip":
        c = K.compress_channel(state["x"], state["plan"], state["bits"], state["group"])
        return c.stored, c.vals, c.scales, K.decompress_channel(c)
    y = state["mod"](*state["inputs"])
    return (y.detach(),) + torch.autograd.grad(y, state["wanted"], state["g"], allow_unused=True)


# ---- what it cannot do without ---------------------------------------------------------------------------------------
def _saved(case, width, bits, group):
    """bytes a token of one saved activation takes: codes, outliers, scales"""
    if case.get("mode") == "ref":
        return width * bits // 8 + 6 * 0.01 * width    # outlier elements of both signs: int32 column and bf16 value
    return width * bits // 8 + 2 * K.num_outlier_channels(width, 0.01) + 2 * (width // group)


def work(case):
    op = case["op"]
    if op == "round_trip":
        m, h = case["tokens"], case["width"]
        return dict(bytes=m * (4 * h + 2 * _saved(case, h, case["bits"], case["group"])), flops=10 * m * h)
    if op == "softmax":
        n = case["batch"] * case["heads"] * case["seq"] ** 2
        return dict(bytes=n * (2 + 2 + 2 + 2 + 2 * 0.06), flops=10 * n)
    if op == "layer":
        b, s, h, i, r = case["batch"], case["seq"], case["hidden"], case["inner"], case["rank"]
        m, base, lora = b * s, 4 * h * h + 3 * h * i, r * (11 * h + 3 * i)
        attention = 2 * b * s * s * h // 2             # one causal product of all heads
        site = lambda n, bits: 2 * _saved(case, n, bits, 128)
        saved = 5 * site(h, case["bits"]) + 3 * site(i, case["bits"]) + 3 * site(h, 8) + site(i, 8)
        return dict(bytes=2 * base * 0.53 + 4 * m * 2 * h + m * saved + 4 * lora,
                    flops=4 * m * base + 6 * m * lora + 7 * attention)
    m, h = case["batch"] * case["seq"], case["width"]
    saved = _saved(case, h, case["bits"], case["group"])
    if op == "linear":
        n = case["out"]
        return dict(bytes=m * (4 * h + 4 * n + 2 * saved) + 6 * n * h, flops=6 * m * n * h)
    if op == "gated":
        return dict(bytes=m * (12 * h + 6 * saved), flops=30 * m * h)
    return dict(bytes=m * (8 * h + 2 * saved), flops=20 * m * h)


# ---- how far another correct implementation may be off -----------------------------------------------------------------
def tolerance(case):
    """about four times what an evaluation of the same formulas in 64 bits differs by from the bf16 results"""
    op = case["op"]
    if op == "round_trip":
        return "exact"                                 # codes, scales and outlier values are defined bit for bit
    if op == "layer":
        # a product summed in another order moves bf16 values by an ulp, and of the 4-bit codes made from them a few by
        # a whole step: gradients differ by 0.5 to 2.4 % between the library's GEMMs / attention and their fp32 forms
        return dict(rel=0.03, max=0.95)
    if op == "gated":
        return dict(rel=2e-2, max=0.95)                # the derivative of act is a chain of bf16 roundings
    if op in ("silu", "gelu"):
        return dict(rel=1.5e-2, max=0.25)              # the same chain
    if op == "softmax":
        return dict(rel=1e-2, max=0.2)
    return dict(rel=7e-3, max=2e-2)
