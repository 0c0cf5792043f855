"""Every form of the products over few tokens against 64 bits, over reductions in which a wave has several blocks: the next one is on its way
while one is used, and the last is asked for twice.  What lies behind a result stays as it was."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def near(got, want, size, extra=0.0):
    """one rounding to bf16 of the result (`extra`: of what was rounded before), and an fp32 sum: an error of 2^-24 of the terms' magnitudes
    for each term, of random sign"""
    bound = 2.0 ** -8 * (want.abs() + extra) + 64 * 2.0 ** -24 * size + 1e-30
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() / bound).max())


# Tokens: one to five tiles a workgroup, and more than one block of them with the last one cut.  Features: one tile a workgroup (16, 64), two
# (4112, the last cut) and four (from 8208 on, 2064 over 257 tokens, 2608 over 400), those from the codes in workgroups of eight waves up to 256
# workgroups, else of four.  24 blocks of 64 are three a wave of eight and six a wave of four; 25, 27 and 33 leave some waves one more.
SHAPES = [(M, N, 64 * blocks) for M, N in ((1, 16), (17, 64), (33, 4112), (80, 4112), (5, 8208), (17, 8208), (33, 8208), (65, 8208), (157, 8208), (129, 11280),
                                           (81, 11264), (5, 16400), (257, 2064), (400, 2608))
          for blocks in (24, 27)] + [(161, 8208, 64 * 25), (96, 11264, 64 * 33)]


@pytest.mark.parametrize("M,N,Kf", SHAPES)
def test_dx(K, M, N, Kf):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    a, b, room = mk(M, Kf), mk(N, Kf), torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")

    def run(out):
        K.check(K._abi.load().hyc_few_rows(a.data_ptr(), Kf, M, Kf, b.data_ptr(), N, out.data_ptr(), K._stream()))
        return out[:M]
    y = run(room)
    near(y, a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t())
    assert (room[M] == 7).all()
    first = y.clone()
    a[M // 2, Kf - 1], b[N // 3, 0] = float("inf"), float("nan")          # (in the last block of the reduction, and in the first)
    y = run(room)
    rows, cols = torch.arange(M, device="cuda") != M // 2, torch.arange(N, device="cuda") != N // 3
    assert torch.equal(y[rows][:, cols], first[rows][:, cols]) and y[:, N // 3].isnan().all() and not y[M // 2].isfinite().any() and (room[M] == 7).all()


@pytest.mark.parametrize("M,N,Kf", SHAPES)
@pytest.mark.parametrize("r", [16, 24])
def test_base_product_with_its_rank_term(K, M, N, Kf, r):
    gen = torch.Generator(device="cuda").manual_seed(M + N + r)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    outs, s = ([N - 16, 16] if N > 16 else [N]), 1.5
    n, q, x, B, h = len(outs), K.nf4_quantize(mk(N, Kf)), mk(M, Kf), [mk(o, r) for o in outs], mk(M, len(outs) * r)
    room = torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")

    def run():
        K.check(K._abi.load().hyc_few_rows_nf4(x.data_ptr(), Kf, M, Kf, q.packed.data_ptr(), q.absmax.data_ptr(), h.data_ptr(), K._ptrs(B), K._i64s(outs), n, r,
                                               s, room.data_ptr(), K._stream()))
        return room[:M]
    y, W = run(), K.nf4_dequantize(q).double()
    up = torch.cat([s * (h[:, i * r:(i + 1) * r].double() @ b.double().t()) for i, b in enumerate(B)], 1)
    near(y, x.double() @ W.t() + up, x.double().abs() @ W.abs().t() + up.abs(), up.abs())
    assert (room[M] == 7).all()
    # an infinity in one token, and in one token's h, reach those tokens and no other
    first, other = y.clone(), (M // 2 + 1) % M
    x[M // 2, Kf - 1], h[other, 0] = float("inf"), float("-inf")
    y = run()
    rows = torch.ones(M, dtype=torch.bool, device="cuda")
    rows[[M // 2, other]] = False
    assert torch.equal(y[rows], first[rows]) and not y[M // 2].isfinite().any() and (room[M] == 7).all()
    assert not y[other, :outs[0]].isfinite().any() and (M == 1 or torch.equal(y[other, outs[0]:], first[other, outs[0]:]))
