"""The fused gated product over the launch shapes its rules choose between: a call over many rows against calls of 200 rows (at most one
row a workgroup), bit for bit - no row knows of another."""
import pytest
import torch

from conftest import bits_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


# 2-bit codes of one to four waves a row, of six, seven and eight (the variant of 512 threads); 4-bit codes of five to eight; both
# sides of 8192 rows and of 32 768
@pytest.mark.parametrize("act,H,bits,group,M", [("silu", 2048, 2, 64, 600), ("silu", 4096, 2, 64, 600), ("gelu", 6144, 2, 64, 300), ("silu", 8192, 2, 64, 601),
                                                ("silu", 11008, 2, 64, 301), ("gelu", 13824, 2, 64, 290), ("silu", 16384, 2, 128, 270),
                                                ("silu", 5120, 4, 128, 600), ("gelu", 7168, 4, 128, 300), ("silu", 8192, 4, 128, 300),
                                                ("silu", 5120, 4, 128, 8400), ("silu", 10240, 2, 64, 8400), ("silu", 5120, 4, 64, 32800)])
def test_rows_are_independent(K, act, H, bits, group, M):
    gen = torch.Generator(device="cuda").manual_seed(H + M)
    mk = lambda: torch.randn(M, H, generator=gen, device="cuda").bfloat16()
    gate, up, g = mk(), mk(), mk()
    plans = [K.select_channels(K.channel_absmax(t[:200]), 11) for t in (gate, up, g)]
    h, *saved = K.gated_act_fwd(act, gate, up, *plans, bits, group)
    grads = K.gated_act_bwd(act, g, *saved)
    for lo in range(0, M, 200) if M < 1000 else (0, 4200, M - 200):
        rows = slice(lo, min(M, lo + 200))
        h1, *saved1 = K.gated_act_fwd(act, gate[rows], up[rows], *plans, bits, group)
        assert bits_equal(h1, h[rows])
        for c, c1 in zip(saved, saved1):
            assert torch.equal(c1.stored, c.stored[rows]) and bits_equal(c1.vals, c.vals[rows]) and bits_equal(c1.scales, c.scales[rows])
        for d, d1 in zip(grads, K.gated_act_bwd(act, g[rows], *saved1)):
            assert bits_equal(d1, d[rows])
