"""Rows of more than 1024 chunks per segment, which several workgroups share: codes, scales, kept values and the restored rows equal the
oracle's bit for bit, and the activation backward from the codes equals the one from the restored rows, at the edges of the rule (1024 chunks and one group more), at shares that do not come out even, with a last share of
one group, with more kept channels than one workgroup has lanes, and with more rows than workgroups."""
import pytest
import torch

from conftest import bits_equal
from oracle import hyc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


@pytest.mark.parametrize("rule", ["absmax", "range"])
@pytest.mark.parametrize("bits,group,M,H,k", [
    (8, 128, 9, 8192, 80),            # 1024 chunks: one workgroup a row
    (8, 128, 9, 8192 + 128, 80), (8, 64, 9, 8192 + 64, 80),
    (8, 128, 2700, 11008, 110),       # more rows than workgroups
    (8, 64, 5, 13824, 2500),          # more kept channels than chunks in a row
    (8, 128, 3, 8192 * 2 + 128, 3), (8, 64, 3, 8192 * 3 + 64, 1), (8, 128, 1, 65536, 0),
    (4, 128, 3, 16384 + 256, 7), (4, 64, 2, 65536, 700), (2, 64, 2, 65536, 70),
    (8, 32, 4, 11008, 9), (1, 64, 2, 65536, 5),   # still walked in turns
])
def test_wide_rows(K, bits, group, M, H, k, rule):
    gen = torch.Generator().manual_seed(bits + H + M)
    x = torch.randn(M, H, generator=gen)
    x[:, torch.randperm(H, generator=gen)[:max(k, 1)]] *= 30.0
    x = x.bfloat16()
    x[0, :group] = 0
    x[0, -group:] = 1.5
    idx = O.hyc_select_channels(O.hyc_channel_scores(x), k)
    xd = x.cuda()
    c = K.compress_channel(xd, K.select_channels(K.channel_absmax(xd), k, rule), bits, group)
    vals, stored, scales = O.hyc_compress(x, idx, bits, group, rule)
    assert bits_equal(c.scales.cpu(), scales) and bits_equal(c.vals.cpu(), vals) and torch.equal(c.stored.cpu(), stored)
    assert bits_equal(K.decompress_channel(c).cpu(), O.hyc_decompress(vals, stored, idx, scales, bits, group))


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("bits,group,M,H,k", [
    (8, 128, 3, 8192, 5), (8, 64, 5, 8192 + 64, 60), (8, 128, 900, 11008, 110), (8, 64, 133, 13824, 2500), (8, 64, 3, 8192 * 3 + 64, 1),
    (8, 128, 2, 65536, 0), (4, 128, 130, 16384 + 256, 7), (2, 64, 2, 65536, 70),
])
def test_activation_backward_of_wide_rows(K, bits, group, M, H, k, act):
    gen = torch.Generator().manual_seed(bits + H + M)
    x = (2 * torch.randn(M, H, generator=gen)).bfloat16().cuda()
    g = torch.randn(M, H, generator=gen).bfloat16().cuda()
    c = K.compress_channel(x, K.select_channels(K.channel_absmax(x), k), bits, group)
    dx = K.act_bwd(act, g, c)
    xh = K.decompress_channel(c)                                 # (a dense source takes the kernel that walks rows in turns)
    assert bits_equal(dx, K.act_bwd(act, g, xh))
    c2 = K.compress_channel(g, K.select_channels(K.channel_absmax(g), k), bits, group)
    for got, want in zip(K.hadamard_bwd(g, c, c2), K.hadamard_bwd(g, xh, K.decompress_channel(c2))):
        assert bits_equal(got, want)
