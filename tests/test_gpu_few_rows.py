"""The products of a LoRA group with its base weight over few tokens, in one launch each, against the same in 64 bits: tokens around a tile
of 16 and a workgroup's five, reductions of one block of 64, of fewer blocks than waves and of an odd number, features in one and two tiles a
workgroup with the last one cut."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def near(got, want, size, roundings):
    """`roundings` to bf16 of the result, and an fp32 sum: an error of 2^-24 of the terms' magnitudes for each term, of random sign"""
    bound = roundings * 2.0 ** -8 * want.abs() + 64 * 2.0 ** -24 * size + 1e-30
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() / bound).max())


@pytest.mark.parametrize("M", [1, 15, 16, 17, 79, 81, 160, 161, 257])
@pytest.mark.parametrize("Kf,outs,r", [(64, [16], 8), (192, [48, 16], 16), (576, [272, 16, 32], 24), (1088, [64], 32), (128, [8208], 16), (128, [4784], 8)])
def test_base_product_with_its_rank_term(K, M, Kf, outs, r):
    n, N, s = len(outs), sum(outs), 1.5
    if not K._abi.load().hyc_few_rows_covers(M, Kf, N, 0):
        pytest.skip("left to the library")
    gen = torch.Generator(device="cuda").manual_seed(M + Kf)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    q, B, h, wide = K.nf4_quantize(mk(N, Kf)), [mk(o, r) for o in outs], mk(M, n * r), mk(M, Kf + 8)
    y = K.few_rows_base(wide[:, :Kf], q, h, B, s, outs)                     # rows with a pitch of their own
    x, W = wide[:, :Kf].double(), K.nf4_dequantize(q).double()
    up = torch.cat([s * (h[:, i * r:(i + 1) * r].double() @ b.double().t()) for i, b in enumerate(B)], 1)
    size = x.abs() @ W.abs().t() + up.abs()
    near(y, x @ W.t() + up, size + 2.0 ** 24 / 64 * 2.0 ** -8 * up.abs(), 1)   # the rank term is rounded by itself: 2^-8 of it at most
    again = K.few_rows_base(x.to(BF16), q, h, B, s, outs)
    assert torch.equal(y, again)
    # a token's result does not depend on the others, but for the tiles they share out among the waves: the same here
    assert torch.equal(K.few_rows_base(wide[:, :Kf], q, h, [torch.zeros_like(b) for b in B], s, outs),
                       K.few_rows_base(wide[:, :Kf], q, torch.zeros_like(h), B, s, outs))


@pytest.mark.parametrize("M", [1, 16, 17, 80, 81, 161, 400])
@pytest.mark.parametrize("Kf,N", [(64, 16), (192, 64), (1088, 80), (128, 8208), (512, 512), (128, 4784), (64, 2608)])
def test_product(K, M, Kf, N):
    if not K._abi.load().hyc_few_rows_covers(M, Kf, N, 1):
        pytest.skip("left to the library")
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    a, b = mk(M, Kf), mk(N, Kf)
    guard = torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")
    assert K.few_rows(guard[:M], a, b)
    near(guard[:M], a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t(), 1)
    assert (guard[M] == 7).all()
    if M > 1:                                               # an infinity and a NaN stay in their row and their column
        a[1, 3], b[5, 2] = float("inf"), float("nan")
        out = torch.empty_like(guard[:M])
        assert K.few_rows(out, a, b)
        rows, cols = torch.arange(M, device="cuda") != 1, torch.arange(N, device="cuda") != 5
        assert torch.equal(out[rows][:, cols], guard[:M][rows][:, cols]) and out[:, 5].isnan().all() and not out[1].isfinite().any()


def test_what_is_left_to_the_library(K, hyc):
    covers = K._abi.load().hyc_few_rows_covers
    assert covers(157, 2048, 11264, 0) and covers(157, 11264 + 64, 2048, 1) and covers(16, 4096, 22016, 0) and covers(16, 22080, 4096, 1)
    for M, Kf, N, grad in ((4096, 4096, 4096, 0), (4096, 4096, 4096, 1), (2049, 64, 16, 0), (1025, 64, 16, 1), (257, 4096, 4096, 1), (0, 64, 16, 0), (8, 96, 16, 0), (8, 64, 24, 1),
                           (64, 1 << 24, 16, 0), (16, 64, 1 << 24, 1)):
        assert not covers(M, Kf, N, grad)
    mk = lambda *shape: torch.randn(*shape, device="cuda").to(BF16)
    q, h = K.nf4_quantize(mk(48, 64)), mk(8, 32)
    B = [mk(16, 16), mk(32, 16)]
    assert K.few_rows_base(mk(8, 64), q, h, B, 1.0, [16, 32]) is not None
    assert K.few_rows_base(mk(8, 72)[:, 1:65], q, h, B, 1.0, [16, 32]) is None          # an odd offset
    assert K.few_rows_base(mk(8, 64), q, h, B, 1.0, [24, 24]) is None                   # a tile of 16 features in two projections
    assert K.few_rows_base(mk(8, 64), K.NF4Weight(q.packed[:-32], q.absmax, q.shape), h, B, 1.0, [16, 32]) is None
    with pytest.raises(ValueError):
        K.few_rows_base(mk(8, 64), q, h, B[::-1], 1.0, [16, 32])
    assert not K.few_rows(mk(8, 16), mk(8, 64), mk(64, 16).t())


@pytest.mark.parametrize("M", [33, 400])
def test_group_under_capture(K, hyc, M):
    """forward and backward of a group in a graph, replayed between eager work of the program's own"""
    import importlib
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    mod = DL.LoRAProjections(256, [128, 64], DL.LayerConfig(hidden=256, lora_r=16), "cuda")
    x, gs = torch.randn(M, 256, device="cuda").to(BF16), [torch.randn(M, o, device="cuda").to(BF16) for o in (128, 64)]
    x.requires_grad_(True)
    leaves = [x, *mod.parameters()]
    step = lambda: [*(ys := mod(x)), *torch.autograd.grad(ys, leaves, gs)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for seed in range(4):
        with torch.no_grad():
            x.copy_(torch.randn(M, 256, device="cuda"))
        graph.replay()
        want = step()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
