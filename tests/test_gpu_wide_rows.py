"""Rows of more than 1024 chunks per segment, which several workgroups share: codes, scales, kept values and the restored rows equal the
oracle's bit for bit at the edges of the rule (1024 chunks and one group more), at shares that do not come out even, with a last share of
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
    (8, 128, 3, 768 * 8 * 2 + 128, 3), (8, 64, 3, 768 * 8 * 3 + 64, 1), (8, 128, 1, 65536, 0),
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
