"""The native host path against the interpreted one: the same launches, so the same bits, for every form either of them takes, and the
same errors for what neither does."""
import importlib

import pytest
import torch

from conftest import bits_equal

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


class Counted:
    """the native functions, with the calls they took"""
    def __init__(self, native):
        self.native, self.taken = native, []

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self.native, name)(*args)
            if out is not None:
                self.taken.append(name)
            return out
        return call


class Off:
    def __getattr__(self, name):
        return lambda *args: None


def both(K, make, *expected):
    """make() -> outputs, natively and interpreted, from the same seeds; `expected`: the native functions that must have run"""
    results, native = [], K.native
    try:
        for K.native in (Counted(native), Off()):
            torch.manual_seed(7)
            results.append([t for t in make() if t is not None])
            if isinstance(K.native, Counted):
                taken = set(K.native.taken)
    finally:
        K.native = native
    assert len(results[0]) == len(results[1])
    for a, b in zip(*results):
        assert a.stride() == b.stride() or a.numel() <= 1
        assert bits_equal(a, b)
    assert taken == set(expected), (taken, expected)


def activation(*shape):
    x = torch.randn(*shape, device="cuda")
    x[..., 3] *= 20
    return x.to(BF16)


def steps(mod, inputs, n=4):
    """outputs and gradients of the calibrated steps of a module"""
    out = []
    for i in range(n):
        y = mod(*inputs)
        if i >= 2:
            leaves = [t for t in inputs if t.requires_grad] + [p for p in mod.parameters()]
            g = torch.randn(y.shape, device="cuda").to(y.dtype)
            out += [y.detach()] + list(torch.autograd.grad(y, leaves, g, allow_unused=True))
    return out


@pytest.mark.parametrize("bits,group", [(2, 64), (4, 128), (8, 128)])
@pytest.mark.parametrize("M", [1, 37])
def test_round_trip(K, bits, group, M):
    def make():
        wide = activation(M, 2048)
        for x in (wide, wide[:, 512:1536], wide[:, :1024].contiguous()):
            plan = K.select_channels(K.channel_absmax(x), 11)
            c = K.compress_channel(x, plan, bits, group)
            yield from (c.stored, c.vals, c.scales, K.decompress_channel(c))
    both(K, make, "compress", "decompress")


@pytest.mark.parametrize("kind", ["rms", "rms_fp32", "gemma", "layer", "layer_plain"])
@pytest.mark.parametrize("shape", [(45, 1024), (2, 9, 1024), (1, 3, 2, 1024)])
def test_norms(K, hyc, kind, shape):
    ops = hyc.operators
    how = dict(sub_outlier_ratio=1.0, sub_outlier_bit=4, rank=0, mode="hyc", group_size=128)

    def make():
        cls = {"rms": ops.EfficientMemoryRMSNorm, "rms_fp32": ops.EfficientMemoryRMSNorm, "gemma": ops.EfficientMemoryRMSNormGemma}
        mod = cls.get(kind, ops.EfficientMemoryLayerNorm)(1024, bias=kind == "layer", **how).cuda()
        mod = mod if kind == "rms_fp32" else mod.to(BF16)
        return steps(mod, [activation(*shape).requires_grad_(True)])
    both(K, make, *{"gemma": (), "layer": ("norm_fwd", "norm_bwd", "bias_grad")}.get(kind, ("norm_fwd", "norm_bwd")))


def test_strided_and_wide_inputs_take_the_interpreted_form(K, hyc):
    """a transposed input, a gradient broadcast from one row, an fp32 gradient"""
    def make():
        mod = hyc.operators.EfficientMemoryRMSNorm(1024, bias=False, sub_outlier_ratio=1.0, sub_outlier_bit=4, rank=0, mode="hyc").cuda().to(BF16)
        x = activation(6, 5, 1024).transpose(0, 1).requires_grad_(True)
        for _ in range(3):
            y = mod(x)
        yield y.detach()
        yield from torch.autograd.grad(y, [x, mod.weight], torch.randn(1, 1, 1024, device="cuda").to(BF16).expand(5, 6, 1024))
    both(K, make)


@pytest.mark.parametrize("method,rank", [("per-channel", 2), ("per-token", 0), ("per-tensor", 0)])
@pytest.mark.parametrize("kind", ["rms", "layer", "silu", "gelu"])
def test_reference_scheme(K, hyc, kind, method, rank):
    ops = hyc.operators
    how = dict(sub_outlier_ratio=1.0, sub_outlier_bit=8, sub_outlier_quantize_method=method, rank=rank)

    def make():
        mod = {"rms": lambda: ops.EfficientMemoryRMSNorm(512, bias=False, **how), "layer": lambda: ops.EfficientMemoryLayerNorm(512, **how),
               "silu": lambda: ops.EfficientMemorySiLU(**how), "gelu": lambda: ops.EfficientMemoryGELU(**how)}[kind]().cuda().to(BF16)
        return steps(mod, [activation(2, 24, 512).requires_grad_(True)], n=5)
    # (an interpreted activation backward restores through kernels.decompress_threshold)
    both(K, make, "threshold_fwd", *{"rms": ("norm_bwd",), "layer": ("norm_bwd", "bias_grad")}.get(kind, ("act_bwd",)))


@pytest.mark.parametrize("out", [16, 256])
@pytest.mark.parametrize("shape", [(33, 1024), (2, 17, 1024)])
@pytest.mark.parametrize("bias", [False, True])
def test_linear(K, hyc, out, shape, bias):
    def make():
        mod = hyc.operators.EfficientMemoryLinear(1024, out, bias=bias, sub_outlier_ratio=1.0, sub_outlier_bit=2, rank=0, mode="hyc",
                                                  group_size=64).cuda().to(BF16)
        x = activation(*shape).requires_grad_(True)
        got = steps(mod, [x])
        mod.weight.requires_grad_(False)            # a frozen weight: nothing is kept
        y = mod(x)
        return got + [y.detach()] + list(torch.autograd.grad(y, [x], torch.ones_like(y)))
    both(K, make, *(("compress",) if bias else ("linear_fwd", "linear_bwd")))


@pytest.mark.parametrize("kind", ["silu", "gelu", "gated"])
@pytest.mark.parametrize("shape", [(5, 2048), (2, 3, 2048)])
def test_activations(K, hyc, kind, shape):
    ops = hyc.operators

    def make():
        if kind == "gated":
            wide = activation(*shape[:-1], 2 * shape[-1]).requires_grad_(True)
            mod = ops.EfficientMemoryGatedAct("silu", sub_outlier_bit=4, group_size=128)
            for _ in range(3):
                y = mod(wide[..., :shape[-1]], wide[..., shape[-1]:])      # halves of one projection
            return [y.detach()] + list(torch.autograd.grad(y, [wide], torch.randn(y.shape, device="cuda").to(BF16)))
        mod = (ops.EfficientMemorySiLU if kind == "silu" else ops.EfficientMemoryGELU)(sub_outlier_ratio=1.0, sub_outlier_bit=4, rank=0, mode="hyc")
        return steps(mod, [activation(*shape).requires_grad_(True)])
    # (the two calibration calls of the gated product compress by themselves)
    both(K, make, *{"gated": ("compress", "gated_fwd", "gated_bwd")}.get(kind, ("act_fwd", "act_bwd")))


def test_softmax(K, hyc):
    def make():
        return steps(hyc.operators.EfficientMemorySoftmax(0.02), [(2 * torch.randn(1, 3, 40, 256, device="cuda")).to(BF16).requires_grad_(True)], n=5)
    both(K, make, "softmax_fwd", "softmax_bwd")


@pytest.mark.parametrize("attention,compress", [("flash", True), ("eager", True), ("flash", False)])
@pytest.mark.parametrize("heads", [8, 4])
@pytest.mark.parametrize("B,S", [(2, 64), (1, 200)])
def test_decoder_layer(K, hyc, attention, compress, heads, B, S):
    DL = importlib.import_module("hyc-lora_amd.decoder_layer")

    def make():
        layer = DL.DecoderLayer(DL.LayerConfig(hidden=512, heads=heads, head_dim=512 // heads, intermediate=1408, lora_r=8, act_bits=8, linear_bits=8,
                                               act_group=64, attention=attention, compress=compress))
        return steps(layer, [activation(B, S, 512).requires_grad_(True)], n=5)
    if not compress:
        return both(K, make, "lora_forward", "rope_attn_fwd")
    extra = ("attn_bwd",) if attention == "flash" else ("attn_kept", "attn_kept_bwd", "decompress")
    both(K, make, "compress", "norm_fwd", "norm_bwd", "lora_forward", "lora_backward", "gated_fwd", "gated_bwd", "rope_attn_fwd", *extra)


def test_the_same_errors(K):
    x = activation(8, 1024)
    plan = K.select_channels(K.channel_absmax(x), 11)
    other = K.select_channels(K.channel_absmax(activation(8, 2048)), 11)
    c = K.compress_channel(x, plan, 4, 128)
    bad = [lambda: K.compress_channel(x.float(), plan, 4, 128), lambda: K.compress_channel(x.cpu(), plan, 4, 128),
           lambda: K.compress_channel(x[None], plan, 4, 128), lambda: K.compress_channel(x, other, 4, 128), lambda: K.compress_channel(x, plan, 3, 128),
           lambda: K.compress_channel(x, plan, 4, 96), lambda: K.compress_channel(x.t(), plan, 4, 128),
           lambda: K.compress_channel(x, K.ChannelPlan(1024, 11, plan.idx.cpu(), plan.plan), 4, 128),
           lambda: K.compress_channel(x, K.ChannelPlan(1024, 12, plan.idx, plan.plan), 4, 128),
           lambda: K.compress_channel(x, K.ChannelPlan(1024, 11, plan.idx, plan.plan, "none"), 4, 128),
           lambda: K.decompress_channel(K.ChannelCompressed(c.stored, c.vals, c.scales, other, 4, 128, 8, 2049)),
           lambda: K.rmsnorm_bwd(x, K.compress_channel(x[:4].contiguous(), plan, 4, 128), torch.ones(1024, device="cuda"), torch.ones(8, device="cuda"))]
    native = K.native
    for f in bad:
        seen = []
        try:
            for K.native in (native, Off()):
                with pytest.raises(Exception) as e:
                    f()
                seen.append((type(e.value), str(e.value)))
        finally:
            K.native = native
        assert seen[0] == seen[1]
