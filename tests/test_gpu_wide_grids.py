"""Rows that several workgroups share, over many rows: what a row becomes does not depend on how many others there are, that is on how a launch
deals them out (the edges of its rules: 128 and 256 workgroups a part, rounds of 256, one a CU over all parts, rows walked in turns)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


@pytest.mark.parametrize("bits,H,M", [(8, 8192 + 64, m) for m in (159, 160, 447, 448, 767, 768, 1023, 1024, 2049)] + [
    (8, 16384 + 64, 341), (8, 16384 + 64, 342), (8, 24576 + 128, 255), (8, 24576 + 128, 256), (8, 32768, 1007), (8, 32768, 1008), (8, 49152, 640),
    (8, 65536, 127), (8, 65536, 128), (8, 65536, 639), (8, 65536, 640), (8, 65536, 1221), (4, 16384 + 128, 448), (4, 65536, 255), (2, 65536, 448)])
def test_a_row_by_itself(K, bits, H, M):
    gen = torch.Generator(device="cuda").manual_seed(M + H)
    x, g = (torch.randn(M, H, generator=gen, device="cuda").to(BF16) for _ in range(2))
    plan = K.select_channels(K.channel_absmax(x), 70)
    every = K.compress_channel(x, plan, bits, 64)
    gelu, mul, xh = K.act_bwd("gelu", g, every), K.hadamard_bwd(g, every, every), K.decompress_channel(every)
    for rows in (slice(0, 50), slice(M // 2 - 3, M // 2 + 4), slice(M - 33, M)):
        c = K.compress_channel(x[rows], plan, bits, 64)
        assert torch.equal(c.stored, every.stored[rows]) and torch.equal(c.vals, every.vals[rows]) and torch.equal(c.scales, every.scales[rows])
        assert torch.equal(K.decompress_channel(c), xh[rows]) and torch.equal(K.act_bwd("gelu", g[rows].contiguous(), c), gelu[rows])
        assert all(torch.equal(a, b[rows]) for a, b in zip(K.hadamard_bwd(g[rows].contiguous(), c, c), mul))
