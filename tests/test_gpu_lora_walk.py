"""dh and dB from one read of dY, at the lengths where the walk over tiles of 32 tokens starts, fills its three or four buffers and ends."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# single tiles, a walk as long as the buffers and one more, ranges of which the last is short, one range for many features
CASES = [(M, outs, r) for r in (8, 16, 32) for M, outs in
         ((1, [8]), (31, [256]), (33, [264, 8]), (97, [72]), (4096 + 1, [4096]), (2048 + 33, [2048, 2048, 1000]), (700, [11008, 11008]), (161, [33000]))]


@pytest.mark.parametrize("M,outs,r", CASES)
def test_both_products_over_the_walk(hyc, M, outs, r):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K, n, total, s = hyc.kernels, len(outs), sum(outs), 1.5
    room = K.lora_room(n, r)
    gen = torch.Generator(device="cuda").manual_seed(M + r)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    B, h, gs = [mk(o, r) for o in outs], mk(M, n * r), [mk(M, o) for o in outs]
    gs[0][-1, -1] = 1e4                                     # (the last element of the last row)

    def close(got, a, b):
        """one rounding to bf16, and an fp32 sum whose error is at most its number of terms x 2^-24 of the sum of their magnitudes (32 for
        terms of random sign)"""
        want, size = s * (a.double() @ b.double()), s * (a.double().abs() @ b.double().abs())
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 32 * 2.0 ** -24 * size + 1e-30).all()

    ext, dh, dB = K.lora_up_bwd(gs, B, h, s, room)
    buf = torch.full_like(ext, float("nan"))
    buf[:, :total] = torch.cat(gs, 1)
    cuts = [sum(outs[:i]) for i in range(n + 1)]
    assert torch.equal(ext[:, :total], buf[:, :total])
    ext2, dh2, dB2 = K.lora_up_bwd([buf[:, a:b] for a, b in zip(cuts, cuts[1:])], B, h, s, room, buf)
    assert torch.equal(ext2, ext) and torch.equal(dh2, dh) and all(torch.equal(a, b) for a, b in zip(dB2, dB))
    for i in range(n):
        close(dh[:, i * r:(i + 1) * r], gs[i], B[i])
        close(dB[i], gs[i].t().contiguous(), h[:, i * r:(i + 1) * r])
    # an infinity reaches its own token's dh and its own feature's dB and nothing else
    gs[0][M // 2, 0] = float("inf")
    _, dh3, dB3 = K.lora_up_bwd(gs, B, h, s, room)
    rows, feats = torch.arange(M, device="cuda") != M // 2, torch.arange(outs[0], device="cuda") != 0
    assert torch.equal(dh3[rows], dh[rows]) and torch.equal(dB3[0][feats], dB[0][feats]) and all(torch.equal(a, b) for a, b in zip(dB3[1:], dB[1:]))
