"""Sums over the tokens (kernels.bias_grad) against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import importlib
    return importlib.import_module("hyc-lora_amd").kernels


# one row; around a round of 32 rows and a block of 256 columns; a last chunk alone; several rounds per block; wide rows
@pytest.mark.parametrize("M,H", [(0, 64), (1, 8), (31, 256), (33, 264), (257, 248), (3627, 1024), (9000, 4104), (40, 16384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bias_grad(K, M, H, dtype):
    gen = torch.Generator().manual_seed(M + H)
    dy = torch.randn(M, H, generator=gen).to(torch.bfloat16)
    got = K.bias_grad(dy.cuda(), dtype).cpu()
    assert got.dtype == dtype and got.shape == (H,)
    want = dy.double().sum(0)
    # every partial sum is at most sum |dy|; each of fewer than M / 8 + 300 additions in a chain rounds by 2^-24 of that
    bound = dy.double().abs().sum(0) * (M / 8 + 300) * 2.0 ** -24
    if dtype == torch.bfloat16:
        bound = bound + want.abs() * 2.0 ** -8
    assert bool(((got.double() - want).abs() <= bound).all())


def test_bias_gradient_of_a_gradient(K):
    """create_graph: the bias gradient can be differentiated with respect to the upstream gradient"""
    import importlib
    ops = importlib.import_module("hyc-lora_amd").operators
    mod = ops.EfficientMemoryLayerNorm(256, mode="hyc", rank=0, group_size=32).cuda().bfloat16()
    x = torch.randn(2, 9, 256, device="cuda").bfloat16()
    for _ in range(3):
        y = mod(x)
    g = torch.randn(2, 9, 256, device="cuda").bfloat16().requires_grad_(True)
    (db,) = torch.autograd.grad(y, [mod.bias], g, create_graph=True)
    (dg,) = torch.autograd.grad(db, [g], torch.arange(256, device="cuda").bfloat16())
    assert torch.equal(dg, torch.arange(256, device="cuda").bfloat16().expand(2, 9, 256))


@pytest.mark.parametrize("M,H", [(3627, 1024), (9700, 13824), (2048, 65536), (16384, 4096)])
@pytest.mark.parametrize("mean", [0.0, 0.05])
def test_bias_grad_rounds_no_more_than_the_plain_sum(K, M, H, mean):
    """in fp32 the error against fp64 (over the whole vector) is that of torch's own fp32 sum or less (5 %: two samples of the
    same size differ by 1 / sqrt(2 H))"""
    gen = torch.Generator(device="cuda").manual_seed(M)
    dy = (mean + 0.02 * torch.randn(M, H, generator=gen, device="cuda")).bfloat16()
    want = dy.double().sum(0)
    error = lambda t: float((t.double() - want).norm() / want.norm())
    assert error(K.bias_grad(dy, torch.float32)) <= 1.05 * error(dy.float().sum(0))
