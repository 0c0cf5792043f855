"""What a natively recorded backward keeps between the passes: tensors, not addresses."""
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
