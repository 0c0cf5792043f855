"""The natively recorded backward of the operators against torch.autograd.Function over the same kernels: the same bits, the same gradients for
whatever is asked of the graph, the same refusals."""
import threading

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


class Watched:
    """the native functions one by one: nothing is recorded past an object in the place of kernels.native"""
    def __init__(self, native):
        self.native = native

    def __getattr__(self, name):
        return getattr(self.native, name)


class Pair(torch.nn.Module):
    """a product of two inputs as a module of one"""
    def __init__(self, product):
        super().__init__()
        self.product = product

    def forward(self, x):
        return self.product(x, x.flip(-1))


def modules(ops):
    hyc = dict(sub_outlier_ratio=1.0, sub_outlier_bit=4, rank=0, mode="hyc", group_size=64)
    ref = dict(sub_outlier_ratio=1.0, sub_outlier_bit=8, sub_outlier_quantize_method="per-channel", rank=2)
    return {"rms": lambda: ops.EfficientMemoryRMSNorm(512, bias=False, **hyc), "layer": lambda: ops.EfficientMemoryLayerNorm(512, **hyc),
            "layer_plain": lambda: ops.EfficientMemoryLayerNorm(512, bias=False, **hyc), "linear": lambda: ops.EfficientMemoryLinear(512, 16, **hyc),
            "linear_wide": lambda: ops.EfficientMemoryLinear(512, 320, **hyc), "silu": lambda: ops.EfficientMemorySiLU(**hyc),
            "gelu": lambda: ops.EfficientMemoryGELU(**hyc), "rms_ref": lambda: ops.EfficientMemoryRMSNorm(512, bias=False, **ref),
            "layer_ref": lambda: ops.EfficientMemoryLayerNorm(512, **ref),
            "gated": lambda: Pair(ops.EfficientMemoryGatedAct("gelu", sub_outlier_bit=4, group_size=64))}


NAMES = {"rms": "_ChannelRMSNormFuncBackward", "layer": "_ChannelLayerNormFuncBackward", "layer_plain": "_ChannelLayerNormFuncBackward",
         "linear": "_ChannelLinearFuncBackward", "linear_wide": "_ChannelLinearFuncBackward", "silu": "_ChannelActFuncBackward",
         "gelu": "_ChannelActFuncBackward", "rms_ref": "_RMSNormFuncBackward", "layer_ref": "EfficientMemoryLayerNormFuncBackward",
         "gated": "_ChannelGatedActFuncBackward"}


def plain(mod, x, g, leaves):
    y = mod(x)
    return [y.detach(), *torch.autograd.grad(y, leaves, g)]


def twice(mod, x, g, leaves):
    y = mod(x)
    return [*torch.autograd.grad(y, leaves, g, retain_graph=True), *torch.autograd.grad(y, leaves, 2 * g)]


def create_graph(mod, x, g, leaves):
    g = g.clone().requires_grad_(True)
    grads = torch.autograd.grad(mod(x), leaves, g, create_graph=True)
    out = [t.detach() for t in grads] + [torch.tensor([t.requires_grad for t in grads])]
    for t in grads:
        if t.requires_grad:
            out += [d for d in torch.autograd.grad(t.float().sum(), [g, *leaves], allow_unused=True, retain_graph=True) if d is not None]
    return out


def batched(mod, x, g, leaves):
    return list(torch.autograd.grad(mod(x), leaves, torch.stack([g, 3 * g]), is_grads_batched=True))


def broadcast(mod, x, g, leaves):
    return list(torch.autograd.grad(mod(x), leaves, g[:1, :1].expand(g.shape)))


def transposed(mod, x, g, leaves):
    return list(torch.autograd.grad(mod(x), leaves, g.transpose(0, 1).contiguous().transpose(0, 1)))


def transposed_input(mod, x, g, leaves):
    x = x.detach().transpose(0, 1).contiguous().transpose(0, 1).requires_grad_(True)
    return list(torch.autograd.grad(mod(x), [x, *leaves[1:]], g))


def half_gradient(mod, x, g, leaves):
    return list(torch.autograd.grad(mod(x).float(), leaves, g.float()))


def undefined(mod, x, g, leaves):
    """a gradient that never comes stands for zeros"""
    class Nothing(torch.autograd.Function):
        @staticmethod
        def forward(ctx, y):
            return y.clone()

        @staticmethod
        def backward(ctx, g):
            return None
    return list(torch.autograd.grad(Nothing.apply(mod(x)), leaves, g, allow_unused=True))


def frozen_weight(mod, x, g, leaves):
    [p.requires_grad_(False) for p in mod.parameters()]
    y = mod(x)
    return [y.detach(), *torch.autograd.grad(y, [x], g)]


def frozen_input(mod, x, g, leaves):
    y = mod(x.detach())
    return [y.detach()] + ([*torch.autograd.grad(y, leaves[1:], g)] if y.requires_grad else [])


def without_gradients(mod, x, g, leaves):
    with torch.no_grad():
        y = mod(x)
    assert not y.requires_grad and y.grad_fn is None
    return [y]


def inference(mod, x, g, leaves):
    with torch.inference_mode():
        return [mod(x.detach()).clone()]


def hooks(mod, x, g, leaves):
    seen, y = [], mod(x)
    y.register_hook(lambda t: 2 * t)
    y.grad_fn.register_hook(lambda into, out: seen.extend(t.clone() for t in into if t is not None))
    y.grad_fn.register_prehook(lambda out: tuple(t if t is None else 3 * t for t in out))     # (a Function's other results have none)
    grads = torch.autograd.grad(y, leaves, g)
    return [*grads, *seen]


def accumulated(mod, x, g, leaves):
    for _ in range(2):
        mod(x).backward(g)
    out = [t.grad.clone() for t in leaves]
    for t in leaves:
        t.grad = None
    return out


def in_place_on_the_output(mod, x, g, leaves):
    """(a Function refuses it where its result is a view of what it computed, or one of several)"""
    y = mod(x)
    try:
        y.mul_(2)
    except RuntimeError:
        assert isinstance(y.grad_fn, torch.autograd.function.BackwardCFunction)
        y = 2 * mod(x)
    return [y.detach(), *torch.autograd.grad(y, leaves, g)]


def other_thread(mod, x, g, leaves):
    got, y = [], mod(x)
    t = threading.Thread(target=lambda: got.extend(torch.autograd.grad(y, leaves, g)))
    t.start()
    t.join()
    return got


def side_stream(mod, x, g, leaves):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y = mod(x)
    torch.cuda.current_stream().wait_stream(s)
    out = [y.detach(), *torch.autograd.grad(y, leaves, g)]
    torch.cuda.synchronize()
    return out


def checkpointed(mod, x, g, leaves):
    from torch.utils.checkpoint import checkpoint
    return list(torch.autograd.grad(checkpoint(mod, x, use_reentrant=False), leaves, g))


def autocast_half(mod, x, g, leaves):
    with torch.autocast("cuda", torch.float16):
        y = mod(x)
    return [y.detach(), *torch.autograd.grad(y, leaves, g.to(y.dtype))]


def saved_hooks(mod, x, g, leaves):
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t, lambda t: t):
        y = mod(x)
    return [*torch.autograd.grad(y, leaves, g), torch.tensor(len(packed))]


def tangent(mod, x, g, leaves):
    import torch.autograd.forward_ad as fw
    with fw.dual_level():
        return [mod(fw.make_dual(x.detach(), g.new_ones(x.shape)))]


def transform(mod, x, g, leaves):
    return [torch.func.grad(lambda t: mod(t).float().sum())(x.detach())]


def mapped(mod, x, g, leaves):
    return [torch.func.vmap(mod)(x.detach())]


def what_the_graph_shows(mod, x, g, leaves):
    y = mod(x)
    fn, c = y.grad_fn, y.grad_fn.saved
    c = c[2] if mod.which == "gated" else c
    assert fn.name() == NAMES[mod.which] and y.grad_fn is fn and not hasattr(fn, "nothing_of_the_kind")
    kept = None if hasattr(c, "plan") else int(c.row_ptr[-1])           # (the room behind the last entry holds anything)
    tensors = [c.stored, c.vals[:kept], *([c.scales, c.plan.idx, c.plan.plan] if kept is None else [c.row_ptr, c.cols[:kept], c.scale, c.L, c.R])]
    numbers = [c.bits, c.M, c.H, c.nbytes() if hasattr(c, "plan") else c.threshold]
    return tensors + [torch.tensor(numbers), torch.tensor([f is not None for f, _ in fn.next_functions[:1]])]


FORMS = [plain, twice, create_graph, batched, broadcast, transposed, transposed_input, half_gradient, undefined, frozen_weight, frozen_input, without_gradients,
         inference, hooks, accumulated, in_place_on_the_output, other_thread, side_stream, checkpointed, autocast_half, saved_hooks, tangent, transform,
         mapped, what_the_graph_shows]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f.__name__)
@pytest.mark.parametrize("which", NAMES)
def test_as_a_function_would(K, hyc, which, form):
    native, results, nodes = K.native, [], []
    try:
        for K.native in (native, Watched(native)):
            torch.manual_seed(3)
            mod = modules(hyc.operators)[which]().cuda().to(BF16)
            mod.which = which
            x = torch.randn(3, 7, 512, device="cuda")
            x[..., 5] *= 20
            x = x.to(BF16).requires_grad_(True)
            g = (0.1 * torch.randn(3, 7, mod(x).shape[-1], device="cuda")).to(BF16)
            for _ in range(3):                          # (the reference's scheme sizes its entries from a first calibrated call)
                y = mod(x)
            nodes.append(isinstance(y.grad_fn, torch.autograd.function.BackwardCFunction))
            leaves = [x, *mod.parameters()]
            try:
                results.append((None, form(mod, x, g, leaves)))
            except Exception as e:
                results.append((type(e), []))
    finally:
        K.native = native
    assert nodes == [False, True]                       # recorded natively, and by a Function
    (e0, a), (e1, b) = results
    assert e0 is e1 and len(a) == len(b), (e0, e1, len(a), len(b))
    for s, t in zip(a, b):
        assert (s is None) == (t is None)
        if s is not None:
            assert s.dtype == t.dtype and s.shape == t.shape and bits_equal(s, t)


def test_a_record_goes_with_its_output(K, hyc):
    """nothing but the graph holds what a node keeps"""
    mod = modules(hyc.operators)["rms"]().cuda().to(BF16)
    x = torch.randn(64, 512, device="cuda").to(BF16).requires_grad_(True)
    for _ in range(3):
        y = mod(x)
    del y
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for _ in range(20):
        y = mod(x)
        torch.autograd.grad(y, [x], torch.ones_like(y))
    held = torch.cuda.memory_allocated()
    del y
    assert held > before
    for _ in range(100):                                # (the engine's thread lets go of the last pass' results a little later)
        if torch.cuda.memory_allocated() == before:
            return
        threading.Event().wait(0.02)
    assert torch.cuda.memory_allocated() == before
