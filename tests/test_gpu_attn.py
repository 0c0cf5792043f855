"""The fused causal attention kernels against plain fp32 attention and its autograd gradients, at the sizes where a tile, a
wave or the diagonal ends."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def heads_first(t, heads):
    B, S, H = t.shape
    return t.view(B, S, heads, H // heads).transpose(1, 2).contiguous()


def attention_fp32(q, k, v, heads, scale):
    """(out [B, S, H], lse [B, heads, S]) in fp32; no transposed operand view reaches a batched product"""
    B, S, H = q.shape
    q, k, v = (heads_first(t, heads) for t in (q, k, v))
    mask = torch.full((S, S), float("-inf"), device=q.device).triu(1)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale + mask
    return torch.matmul(torch.softmax(s, -1), v).transpose(1, 2).reshape(B, S, H), torch.logsumexp(s, -1)


def close(got, want, bound, zero=0.0):
    # zero: an element's error where the exact result vanishes
    err = (got.double() - want.double()).norm()
    assert err <= bound * want.double().norm() + zero * math.sqrt(want.numel()), float(err / want.double().norm())


# a walked tile is 64 rows, a wave owns 32, a workgroup 128; 513 and more walk several tiles on both sides of the diagonal; 13
# batches of 8 heads and 5 blocks are more workgroups than two per CU, where the order of the blocks is another
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,S,heads", [(1, 1, 1), (2, 31, 3), (1, 33, 2), (2, 64, 1), (1, 65, 8), (1, 127, 2), (3, 129, 2), (1, 513, 5),
                                       (2, 1030, 2), (13, 513, 8)])
def test_attention_against_fp32(K, hd, B, S, heads):
    H, scale = heads * hd, 1.0 / math.sqrt(hd)
    gen = torch.Generator(device="cuda").manual_seed(S * hd)
    mk = lambda width: torch.randn(B, S, width, generator=gen, device="cuda").bfloat16()
    q, k, g = mk(H), mk(H), mk(H)
    v = mk(2 * H)[..., H:]                                     # a column slice of a wider matrix, as the projections leave it
    out, lse = K.attn_fwd(q, k, v, heads, scale)
    leaves = [t.float().detach().contiguous().requires_grad_(True) for t in (q, k, v)]
    want, want_lse = attention_fp32(*leaves, heads, scale)
    # probabilities are rounded to bf16 for the second product and the result once more; a rounding is 2^-8 / sqrt(3) of the
    # leading binade in the root mean square, below 2^-9 over a norm
    close(out, want.detach(), 2 * 2.0 ** -9)
    assert (lse - want_lse.detach()).abs().max() < 1e-4        # fp32 sums of at most 1030 terms
    grads = torch.autograd.grad(want, leaves, g.float())
    # P or dS, the stored output inside delta, and the result: three such roundings
    # (a single query attends to itself alone and its dq and dk vanish: fp32 sums of hd products in two orders, about 1e-6 each)
    for got, ref in zip(K.attn_bwd(g, q, k, v, out, lse, heads, scale), grads):
        close(got, ref, 3 * 2.0 ** -9, 1e-5 if S == 1 else 0.0)


@pytest.mark.parametrize("hd,S", [(128, 77), (64, 200)])
def test_attention_gradients_before_the_rotation(K, hd, S):
    """cos / sin turn dq and dk into the gradients of the unrotated tensors: the same bits as rotating them back afterwards,
    up to the one rounding that is saved"""
    B, heads = 2, 3
    H, scale = heads * hd, 0.1
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v, g = (torch.randn(B, S, H, generator=gen, device="cuda").bfloat16() for _ in range(4))
    ang = torch.rand(S, hd, generator=gen, device="cuda") * 6.28
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    out, lse = K.attn_fwd(q, k, v, heads, scale)
    plain = K.attn_bwd(g, q, k, v, out, lse, heads, scale)
    turned = K.attn_bwd(g, q, k, v, out, lse, heads, scale, cos, sin)
    for a, b in zip(plain[:2], turned[:2]):
        want = K.rope_from_heads(heads_first(a, heads), cos, sin)
        close(b, want, 2 * 2.0 ** -9)
    assert torch.equal(plain[2], turned[2])


@pytest.mark.parametrize("hd", [64, 128])
def test_attention_stays_inside_its_batch_element(K, hd):
    """rows of the tiles past a batch element's end must not reach its results, whatever lies there"""
    S, heads = 70, 2
    H = heads * hd
    gen = torch.Generator(device="cuda").manual_seed(9)
    q, k, v, g = (torch.randn(2, S, H, generator=gen, device="cuda").bfloat16() for _ in range(4))
    alone = [t[:1].clone() for t in (q, k, v, g)]
    for t in (q, k, v, g):
        t[1] = float("nan")
    o1, l1 = K.attn_fwd(*alone[:3], heads, 0.1)
    o2, l2 = K.attn_fwd(q, k, v, heads, 0.1)
    assert torch.equal(o1[0], o2[0]) and torch.equal(l1[0], l2[0])
    for a, b in zip(K.attn_bwd(alone[3], *alone[:3], o1, l1, heads, 0.1), K.attn_bwd(g, q, k, v, o2, l2, heads, 0.1)):
        assert torch.equal(a[0], b[0])


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("scale", [0.1, 3.0])
@pytest.mark.parametrize("dead", [64, 130])
def test_scores_of_minus_infinity_have_no_weight(K, hd, scale, dead):
    """whole tiles of keys that score -inf: later queries attend to the keys behind them, as in the softmax written out; queries
    that see nothing else are NaN there and here"""
    S, heads = 200, 2
    H = heads * hd
    gen = torch.Generator(device="cuda").manual_seed(10)
    q, k, v = (torch.randn(1, S, H, generator=gen, device="cuda").bfloat16() for _ in range(3))
    q[..., ::hd] = 1.0
    k[:, :dead, ::hd] = float("-inf")
    out, lse = K.attn_fwd(q, k, v, heads, scale)
    want, want_lse = attention_fp32(q.float(), k.float(), v.float(), heads, scale)
    assert torch.isfinite(want[:, dead:]).all()
    close(out[:, dead:], want[:, dead:], 2 * 2.0 ** -9)
    assert (lse[..., dead:] - want_lse[..., dead:]).abs().max() < 1e-4 * max(1.0, scale / 0.1)
    assert out[:, :dead].isnan().all() and (lse[..., :dead] == float("-inf")).all()


def test_attention_refuses_what_it_does_not_cover(K):
    assert not K.attn_supported(32, 64, 128) and not K.attn_supported(128, 1 << 18, 1 << 12)
    q = torch.zeros(1, 8, 64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(NotImplementedError):
        K.attn_fwd(q, q, q, 2, 0.1)
    with pytest.raises(ValueError):
        K.attn_fwd(q, q[:, :4], q, 1, 0.1)
    out, lse = K.attn_fwd(q, q, q, 1, 0.1)
    for scale in (0.0, -0.1):
        with pytest.raises(ValueError):
            K.attn_fwd(q, q, q, 1, scale)
        with pytest.raises(ValueError):
            K.attn_bwd(q, q, q, q, out, lse, 1, scale)
