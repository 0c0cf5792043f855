"""Linear layers of few output features: x w^T and g w by the kernels that serve them, against the products in fp32, at the edges of
their tiles (16 and 128 tokens, 64 channels, 256 features) and on both sides of the line to the library."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def close(got, want):
    """one rounding of an fp32 sum to bf16 (at most 2^-8 of the element), plus the sums' own error (fp32, a few thousand terms)"""
    want = want.double()
    bound = 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max().clamp_min(1e-30)
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() / bound).max())


# (both sides of 3 * 2^24 elements of x with 16 and 24 features, of 2^26 with 32; no multiple of 64, 33 features: the library)
CASES = [((1,), 64, 8), ((16,), 64, 16), ((17,), 128, 24), ((3, 43), 192, 32), ((2, 1, 64), 320, 8), ((127,), 256, 16), ((4, 1025), 4096, 16),
         ((12288,), 4096, 24), ((12289,), 4096, 16), ((16385,), 4096, 32), ((33,), 120, 8), ((33,), 128, 33), ((40,), 1024, 64)]


@pytest.mark.parametrize("shape,Kf,N", CASES)
def test_products(K, hyc, shape, Kf, N):
    gen = torch.Generator(device="cuda").manual_seed(Kf + N)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()
    x, w, g = mk(*shape, Kf), mk(N, Kf), mk(*shape, N)
    M = g.numel() // N
    thin = N <= 32 and Kf % 64 == 0
    with torch.no_grad():
        assert K._thin(x, w, False) == (thin and M * Kf <= 3 << 24) and K._thin(g, w, True) == (thin and (N <= 16 or M * Kf <= 1 << 26))
        y, dx = K.linear_fwd(x, w), K.linear_dx(g, w)
        assert y.shape == g.shape and dx.shape == x.shape and y.is_contiguous() and dx.is_contiguous()
        close(y, x.float() @ w.float().t())
        close(dx, g.float() @ w.float())
        # what lies in one token stays there
        x.view(M, Kf)[M // 2, 5], g.view(M, N)[M // 2, N - 1] = float("inf"), float("nan")
        for got, plain in ((K.linear_fwd(x, w), y), (K.linear_dx(g, w), dx)):
            got, plain = got.view(M, -1), plain.view(M, -1)
            assert not got[M // 2].isfinite().any() and torch.equal(got[:M // 2], plain[:M // 2]) and torch.equal(got[M // 2 + 1:], plain[M // 2 + 1:])


def test_what_the_kernels_do_not_read(K):
    """strided rows, an odd address, a transposed weight, other types, gradients of gradients: torch's product as before"""
    x, w = torch.randn(24, 256, device="cuda").bfloat16(), torch.randn(16, 256, device="cuda").bfloat16()
    odd = torch.empty(24 * 256 + 1, device="cuda", dtype=BF16)[1:].view(24, 256).copy_(x)
    with torch.no_grad():
        assert K._thin(x, w, False)
        for a, b in ((x.repeat(1, 2)[:, :256], w), (odd, w), (x, w.t().contiguous().t()), (x.float(), w.float()), (x[0], w)):
            assert not K._thin(a, b, False)
            close(K.linear_fwd(a, b), a.float() @ b.float().t())
        with pytest.raises(RuntimeError):
            K.linear_fwd(x[:, :128].contiguous(), w)
    g = torch.randn(24, 16, device="cuda").bfloat16().requires_grad_(True)
    assert K.linear_dx(g, w).requires_grad
