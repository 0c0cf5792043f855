"""What a natively recorded backward keeps between the passes: tensors, not addresses."""
import threading
import weakref

import pytest
import torch

from test_gpu_nodes import BF16, NAMES, modules

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def calibrated(hyc, which):
    torch.manual_seed(5)
    mod = modules(hyc.operators)[which]().cuda().to(BF16)
    x = torch.randn(3, 7, 512, device="cuda")
    x[..., 5] *= 20
    x = x.to(BF16).requires_grad_(True)
    for _ in range(3):
        y = mod(x)
    g = (0.1 * torch.randn(y.shape, device="cuda")).to(BF16)
    return mod, x, g, [x, *mod.parameters()]


@pytest.mark.parametrize("which", NAMES)
def test_a_tensor_that_moved_is_read_where_it_lies(K, hyc, which):
    """plans, scales and bases that are given other memory between the forward and the backward pass"""
    mod, x, g, leaves = calibrated(hyc, which)
    want = torch.autograd.grad(mod(x), leaves, g)
    inner = mod.product if which == "gated" else mod
    if which.endswith("_ref"):
        kept = list(inner.static_value[1:])
    else:
        sites = [getattr(inner, s) for s in ("site_act", "site_up", "site_gate")] if which == "gated" else [inner.site]
        kept = [t for s in sites for t in (s.plan.idx, s.plan.plan)]
    y = mod(x)
    old = [t.detach() for t in kept]                        # (the memory they were in: still there, and holds zeros now)
    for t, o in zip(kept, old):
        t.data = t.clone()
        assert t.data_ptr() != o.data_ptr()
        o.zero_()
    got = torch.autograd.grad(y, leaves, g)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def looked_at(fn, which):
    """what a program may do with a Function's context between the passes"""
    c = fn.saved
    fn.note = [1]
    fn.note.append(2)
    assert fn.saved is c and fn.note == [1, 2]
    del fn.note
    assert not hasattr(fn, "note")
    with pytest.raises(AttributeError):
        del fn.note
    first = c[0] if which == "gated" else c
    if hasattr(first, "plan"):
        assert first.plan is first.plan and fn.saved is c
    first.vals = torch.full_like(first.vals, 0.5)            # another tensor in the place of the one that was kept
    fn.needs_input_grad = tuple(fn.needs_input_grad)


@pytest.mark.parametrize("which", NAMES)
def test_a_record_that_was_looked_at_is_a_context(K, hyc, which):
    native, results = K.native, []

    class Watched:
        def __getattr__(self, name):
            return getattr(native, name)
    try:
        for K.native in (native, Watched()):
            mod, x, g, leaves = calibrated(hyc, which)
            plain = torch.autograd.grad(mod(x), leaves, g)
            y = mod(x)
            looked_at(y.grad_fn, which)
            results.append(torch.autograd.grad(y, leaves, g))
            assert not torch.equal(results[-1][1 if len(leaves) > 1 else 0], plain[1 if len(leaves) > 1 else 0])
    finally:
        K.native = native
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_what_was_written_to_a_record_goes_with_it(K, hyc):
    class Thing:
        pass
    mod, x, g, leaves = calibrated(hyc, "rms")
    thing, y = Thing(), mod(x)
    gone = weakref.ref(thing)
    y.grad_fn.thing = thing
    torch.autograd.grad(y, leaves, g)
    del thing
    assert gone() is y.grad_fn.thing
    del y
    for _ in range(100):                                     # (the engine's thread lets go of a pass a little later)
        if gone() is None:
            return
        threading.Event().wait(0.02)
    assert gone() is None
