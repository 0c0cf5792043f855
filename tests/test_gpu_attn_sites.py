"""The saved activations of fused attention taken in one launch each way (csrc/attn_sites.hip), against the kernels that take them one
by one: the same arithmetic in the same order, so the same bits."""
import ctypes
import importlib

import pytest
import torch

from conftest import bits_equal

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


# B, S, heads, head size, bits, group, outlier channels: a row of eight lanes, of a part of a wave, of one and several waves, of more
# than 256 lanes; one row, an odd number, more rows than workgroups; no outliers, chunks of three to eight, more than there are lanes;
# and rows the kernels leave to the general form (segments of half a head)
SHAPES = [(1, 1, 2, 64, 4, 64, 3), (3, 7, 2, 128, 4, 128, 0), (2, 33, 6, 64, 4, 64, 80), (1, 45, 8, 128, 8, 128, 11), (2, 5, 3, 64, 8, 64, 150),
          (1, 300, 32, 64, 4, 128, 21), (1, 2100, 4, 64, 8, 64, 7), (2, 901, 32, 128, 8, 128, 41), (1, 1000, 32, 128, 8, 64, 41),
          (1, 4200, 16, 128, 4, 64, 900),
          (1, 9, 3, 128, 4, 64, 5), (1, 9, 5, 64, 8, 64, 5), (1, 17, 3, 64, 4, 32, 5)]


def tensors(B, S, heads, hd, n, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.randn(B, S, n * heads * hd + 8, device="cuda", generator=gen)
    wide[..., 5::37] *= 25
    wide = wide.to(BF16)
    return [wide[..., i * heads * hd:(i + 1) * heads * hd] for i in range(n)]         # column slices: rows further apart than they are long


@pytest.mark.parametrize("rule", ["absmax", "range"])
@pytest.mark.parametrize("B,S,heads,hd,bits,group,k", SHAPES)
def test_sites(K, hyc, B, S, heads, hd, bits, group, k, rule):
    DL = importlib.import_module("hyc-lora_amd.decoder_layer")
    H, M = heads * hd, B * S
    q, kk, v = tensors(B, S, heads, hd, 3, seed=M + H)
    cos, sin = DL.rope_tables(S, hd, 1e4, "cuda")
    scale = hd ** -0.5
    rows = [K.rope_rows(q, heads, cos, sin), K.rope_rows(kk, heads, cos, sin), v]
    out, lse = K.attn_fwd(rows[0], rows[1], v, heads, scale)
    every = [t.reshape(M, H) for t in (*rows, out)]
    plans = tuple(K.select_channels(K.channel_absmax(t.contiguous()), k, rule) for t in every)
    one_by_one = [K.compress_channel(t, p, bits, group) for t, p in zip(every, plans)]
    for n in (3, 4):
        done = K.native.rope_attn_fwd(q, kk, v, heads, cos, sin, scale, False, plans[:n], bits, group)
        assert all(bits_equal(a, b) for a, b in zip(done[:4], (rows[0], rows[1], out, lse)))
        assert len(done[4]) == n
        for a, b in zip(done[4], one_by_one):
            assert bits_equal(a.stored, b.stored) and bits_equal(a.vals, b.vals) and bits_equal(a.scales, b.scales)

    g = (0.02 * torch.randn(B, S, H, device="cuda")).to(BF16)
    restored = [K.decompress_channel(c).view(B, S, H) for c in one_by_one]
    want = K.attn_bwd(g, *restored, lse, heads, scale, cos, sin)
    got = K.native.attn_bwd(g, list(one_by_one), lse, heads, cos, sin, scale, None)
    assert all(bits_equal(a, b) for a, b in zip(got[:3], want[:3]))

    # the entry itself, and what it says about rows it does not cover
    lib, abi = hyc._abi.load(), hyc._abi
    P = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    xhat = [torch.full((M, H), 7.0, dtype=BF16, device="cuda") for _ in range(3)]
    d = (abi.HycDesc * 3)(*[c.desc() for c in one_by_one[:3]])
    rc = lib.hyc_attn_sites_bwd(P([c.stored for c in one_by_one[:3]]), P([c.vals for c in one_by_one[:3]]), P([c.scales for c in one_by_one[:3]]), d, 3,
                                B, S, heads, hd, P(xhat), None, 0, None, 0.0, None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    covered = (H * bits // 8) % hd == 0 and group in (64, 128)
    assert rc == (0 if covered else abi.ENOTSUP)
    if covered:
        assert all(bits_equal(a.view(B, S, H), b) for a, b in zip(xhat, restored))


def test_arguments_are_judged_before_a_launch(hyc):
    lib, abi = hyc._abi.load(), hyc._abi
    d = (abi.HycDesc * 4)()
    for one in d:
        one.mode, one.bits, one.group, one.chan_plan = abi.MODE_CHANNEL, 4, 64, 1
    fwd = lambda hd, B=1, S=8: lib.hyc_attn_sites_fwd(None, None, None, None, B, S, 2, hd, d, None, None, None, None, None)
    bwd = lambda n, hd=64, B=1, S=8: lib.hyc_attn_sites_bwd(None, None, None, d, n, B, S, 2, hd, None, None, 0, None, 0.1, None, None)
    assert fwd(64) == abi.EFAULT and bwd(3) == abi.EFAULT and fwd(64, B=0) == 0 and bwd(4, S=0) == 0
    assert fwd(96) == abi.ENOTSUP and bwd(3, hd=32) == abi.ENOTSUP and bwd(5) == abi.EINVAL and fwd(64, S=1 << 31) == abi.ENOTSUP
    d[1].bits = 8
    assert fwd(64) == abi.ENOTSUP
    d[1].bits, d[1].mode = 4, abi.MODE_THRESHOLD
    assert bwd(3) == abi.ENOTSUP
