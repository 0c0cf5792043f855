"""hyc_lora_up_bwd at the edges of what its launches count: a range of dY of nearly 2 GiB, and rows of ext that are 1 GiB apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def up_bwd(K, gs, pitches, B, h, scale, ext, ld_ext, room, copy):
    lib, (M, nr), n, outs = K._abi.load(), h.shape, len(B), [b.shape[0] for b in B]
    dh, dB = torch.empty_like(h), [torch.empty_like(b) for b in B]
    ws = torch.empty(lib.hyc_lora_up_bwd_workspace_bytes(M, K._i64s(outs), n, nr // n) // 4, dtype=torch.float32, device="cuda")
    K.check(lib.hyc_lora_up_bwd(K._ptrs(gs), K._i64s(pitches), M, K._i64s(outs), K._ptrs(B), h.data_ptr(), n, nr // n, scale, dh.data_ptr(),
                                ext.data_ptr(), ld_ext, room, copy, K._ptrs(dB), ws.data_ptr(), K._stream()))
    return dh, dB


def close(got, a, b, s):
    """one rounding to bf16, and an fp32 sum whose error is at most its number of terms x 2^-24 of the sum of their magnitudes (32 for
    terms of random sign)"""
    want, size = s * (a.double() @ b.double()), s * (a.double().abs() @ b.double().abs())
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 32 * 2.0 ** -24 * size + 1e-30).all()


@pytest.mark.parametrize("M,out,pitch", [(8386, 127584, 127584 + 64), (65, 71680, 11184816), (98304, 64, 32760)])
def test_a_range_that_fits_in_two(K, M, out, pitch):
    r, room, s = 8, 64, 1.5
    gen = torch.Generator(device="cuda").manual_seed(M)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    B, h = mk(out, r), mk(M, r)
    ext = torch.zeros(M, pitch, dtype=BF16, device="cuda")
    for m in range(0, M, 8192):
        ext[m:m + 8192, :out] = mk(min(8192, M - m), out)
    dh, (dB,) = up_bwd(K, [ext], [pitch], [B], h, s, ext, pitch, room, 0)
    rows = torch.tensor([0, 31, 32, M // 2 - 1, M // 2, M - 1], device="cuda")
    feats = torch.tensor([0, 7, out // 2, out - 1], device="cuda")
    close(dh[rows], ext[rows, :out], B, s)
    close(dB[feats], ext[:, feats].t().contiguous(), h, s)
    assert torch.equal(ext[:, out:out + r], dh) and not ext[:, out + r:out + room].any()


@pytest.mark.parametrize("ld_ext", [(1 << 29) - 8, 1 << 29])
def test_rows_of_ext_far_apart(K, ld_ext):
    M, outs, r, room, s = 3, [264, 8], 16, 64, 1.5
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(BF16)
    gs, B, h, total = [mk(M, o) for o in outs], [mk(o, r) for o in outs], mk(M, 2 * r), sum(outs)
    near, far = (torch.zeros((M - 1) * ld + total + room, dtype=BF16, device="cuda") for ld in (total + room, ld_ext))
    want = up_bwd(K, gs, outs, B, h, s, near, total + room, room, 1)
    got = up_bwd(K, gs, outs, B, h, s, far, ld_ext, room, 1)
    assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[1], want[1]))
    for m in range(M):
        assert torch.equal(far[m * ld_ext:][:total + room], near[m * (total + room):][:total + room])
    assert torch.equal(near.view(M, -1)[:, :264], gs[0]) and torch.equal(near.view(M, -1)[:, 264:272], gs[1])
