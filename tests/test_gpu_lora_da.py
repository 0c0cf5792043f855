"""dA of a LoRA group: however many rows of it a call takes, every element is the sum that calls of up to 32 rows give, bit for bit in fp32."""
import importlib
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def saved(K, x, bits):
    if bits == "dense":
        return x
    plan = K.select_channels(K.channel_absmax(x), K.num_outlier_channels(x.shape[1], 0.01))
    return K.compress_channel(x, plan, bits, 64)


# tokens on both sides of the changes in waves and splits; one projection more than a call takes; ranks that do not divide 32
@pytest.mark.parametrize("bits", [1, 2, 4, 8, "dense"])
@pytest.mark.parametrize("M,H", [(1, 1024), (157, 2048), (1000, 1024), (2048, 4096), (3072, 1024), (4096, 4096), (4100, 2048), (8192, 1024)])
def test_sums_keep_their_order(K, hyc, M, H, bits):
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    gen = torch.Generator(device="cuda").manual_seed(M + H)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    src = saved(K, mk(M, H).to(BF16), bits)
    for n, r in ((3, 16), (2, 32), (3, 32), (3, 24), (4, 32), (3, 8), (5, 32)):
        dh = (0.02 * mk(M, n * r)).to(BF16)
        dA = DL._LoRAProjectionsFunc._grad_A(types.SimpleNamespace(saved_x=src), dh, [torch.empty(r, H, device="cuda")] * n)
        few = max(1, 32 // r) * r
        want = torch.cat([K.gradw_gemm(dh[:, c:c + few], src, out_dtype=torch.float32) for c in range(0, n * r, few)])
        assert len(dA) == n and torch.equal(torch.cat(dA), want)


@pytest.mark.parametrize("M", [157, 2048])
def test_the_native_call_does_the_same(K, hyc, M):
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    mod = DL.LoRAProjections(1024, [256, 128, 64], DL.LayerConfig(hidden=1024, lora_r=16, linear_bits=8), "cuda")
    x = torch.randn(M, 1024, device="cuda").to(BF16).requires_grad_(True)
    gs = [torch.randn(M, o, device="cuda").to(BF16) for o in (256, 128, 64)]
    for B in list(mod.parameters()):
        torch.nn.init.normal_(B, std=0.05)
    mod(x)
    native, results = K.native, []

    class General:
        def __getattr__(self, name):
            return (lambda *a: None) if name == "lora_backward" else getattr(native, name)
    try:
        for K.native in (native, General()):
            ys = mod(x)
            results.append(torch.autograd.grad(ys, list(mod.parameters()), gs))
    finally:
        K.native = native
    assert all(torch.equal(a, b) for a, b in zip(*results))
