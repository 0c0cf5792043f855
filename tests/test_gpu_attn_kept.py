"""Causal attention that keeps its probabilities above a threshold (hyc_attn_kept*) against fp64, at the sizes where a tile, a wave,
the diagonal, a slab row or a round of entries ends."""
import math

import pytest
import torch

from test_gpu_attn import close, heads_first

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def tensors(B, S, heads, hd, gain=1.0):
    gen = torch.Generator(device="cuda").manual_seed(S * hd + heads)
    mk = lambda width: torch.randn(B, S, width, generator=gen, device="cuda")
    H = heads * hd
    return (gain * mk(H)).bfloat16(), mk(H).bfloat16(), mk(2 * H).bfloat16()[..., H:], mk(H).bfloat16()


def probabilities(q, k, heads, scale):
    """(fp64 [B * heads, S, S] softmax(bf16(score)), the scores)"""
    B, S, H = q.shape
    q, k = (heads_first(t, heads).double().flatten(0, 1) for t in (q, k))
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    mask = torch.full((S, S), float("-inf"), device=q.device).triu(1)
    return torch.softmax(s.bfloat16().double() + mask, -1), s


def keep(K, q, k, v, heads, scale, thr, cap, group, share=None):
    out, lse = K.attn_fwd(q, k, v, heads, scale, round_scores=True)
    total, kept, first = q.shape[0] * heads, [], 0
    while first < total:
        n = min(group, total - first)
        budget = None
        if share is not None:                       # room for `share` entries per row
            budget = K.KeptBudget()
            budget.per_row = share
        kept.append(K.attn_kept(q, k, lse, heads, scale, thr, budget, cap, first, n))
        first += n
    return out, kept


# a tile is 64 keys, a wave 32 queries, a workgroup 128 of them and 4 in the gathers; rows of more than 64 entries take several
# rounds there (thr 1e-5 keeps nearly all of a row); caps below a row's entries take the second pass over the scores
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,S,heads,thr,cap,group", [(1, 8, 1, 0.3, 8, 1), (2, 32, 3, 0.05, 16, 4), (1, 72, 8, 0.02, 4, 8), (1, 136, 2, 1e-5, 32, 1),
                                                     (3, 264, 2, 0.01, 64, 5), (1, 520, 8, 1e-3, 16, 8), (1, 1032, 16, 0.004, 64, 16)])
def test_kept_entries_and_gradients(K, hd, B, S, heads, thr, cap, group):
    scale = 1.0 / math.sqrt(hd)
    q, k, v, g = tensors(B, S, heads, hd, gain=2.0)
    out, kept = keep(K, q, k, v, heads, scale, thr, cap, group)
    want, score = probabilities(q, k, heads, scale)
    thr = float(torch.tensor(thr).bfloat16())
    # a probability is rounded for the second product and the result once more; a score that rounds to the other side moves its weight
    # by up to 2^-7 of the score, one in 2^9 of them
    close(heads_first(out, heads).flatten(0, 1), torch.matmul(want, heads_first(v.contiguous(), heads).double().flatten(0, 1)), 2.5 * 2.0 ** -9)
    dense = torch.cat([K.softmax_dense(sp) for sp in kept]).double()
    nnz = 0
    for sp in kept:
        n = int(sp.row_ptr[-1])
        assert n == int(sp.total) <= sp.cols.numel()
        rows = torch.repeat_interleave(torch.arange(sp.rows, device="cuda"), (sp.row_ptr[1:] - sp.row_ptr[:-1]).long())
        cols = sp.cols[:n].long()
        assert bool((cols[1:] > cols[:-1])[rows[1:] == rows[:-1]].all()) and bool((cols <= rows % S).all())
        assert bool((sp.vals[:n].float() > thr).all())
        nnz += n
    assert nnz == int((dense > 0).sum())            # no two entries of a row share a column
    # an entry is rounded to bf16 (2^-8 with the fp32 sums); a score beside the middle of two bf16 values may round to the other of
    # them, 2^-7 of it away, and the set may differ where either takes the exact value across the threshold
    near = 2.0 ** -8 + score.abs() * 2.0 ** -7
    off = ((dense - want).abs() / want)[dense > 0]
    assert bool((off <= near[dense > 0]).all()) and float((off > 2.0 ** -8).double().mean()) < 0.01
    differ = (dense > 0) != (want > thr)
    assert not bool(differ[(want - thr).abs() > thr * near].any()) and int(differ.sum()) <= 1 + 0.01 * nnz
    # gradients at these entries, in fp64
    qh, kh, vh, gh = (heads_first(t, heads).double().flatten(0, 1) for t in (q, k, v.contiguous(), g))
    dp = torch.matmul(gh, vh.transpose(1, 2).contiguous())
    ds = dense * (dp - (dp * dense).sum(-1, keepdim=True))
    back = lambda t: t.view(B, heads, S, hd).transpose(1, 2).reshape(B, S, heads * hd)
    exact = (back(scale * torch.matmul(ds, kh)), back(scale * torch.matmul(ds.transpose(1, 2).contiguous(), qh)),
             back(torch.matmul(dense.transpose(1, 2).contiguous(), gh)))
    for i, (got, ref) in enumerate(zip(K.attn_kept_bwd(g, q, k, v, kept, heads, scale), exact)):
        # dS (dk only) and the result are rounded to bf16: 2^-9 each over a norm; fp32 sums beside them
        close(got, ref, (2 if i == 1 else 1) * 2.0 ** -9, 1e-6)


@pytest.mark.parametrize("hd,S", [(128, 136), (64, 200)])
def test_gradients_before_the_rotation_and_side_by_side(K, hd, S):
    B, heads, room = 2, 3, 64
    H, scale = heads * hd, 0.1
    q, k, v, g = tensors(B, S, heads, hd)
    _, kept = keep(K, q, k, v, heads, scale, 0.01, 32, 6)
    ang = torch.rand(S, hd, device="cuda") * 6.28
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    plain = K.attn_kept_bwd(g, q, k, v, kept, heads, scale)
    turned = K.attn_kept_bwd(g, q, k, v, kept, heads, scale, cos, sin, room=room)
    for a, b in zip(plain[:2], turned[:2]):
        close(b, K.rope_from_heads(heads_first(a, heads), cos, sin), 2 * 2.0 ** -9)
    assert torch.equal(plain[2], turned[2]) and turned[3].shape == (B * S, 3 * H + room)
    for i in range(3):
        assert turned[i].data_ptr() == turned[3].data_ptr() + 2 * i * H


def test_entries_past_the_budget_are_dropped_and_counted(K):
    """offsets cut off at the capacity: what is kept is a prefix of the rows, the total says how many there were, and the gradients
    are those of the kept prefix"""
    B, S, heads, hd, scale = 1, 512, 4, 64, 0.125
    q, k, v, g = tensors(B, S, heads, hd)
    _, (full,) = keep(K, q, k, v, heads, scale, 1e-3, 64, heads)
    out, lse = K.attn_fwd(q, k, v, heads, scale, round_scores=True)
    budget = K.KeptBudget()
    budget.per_row = 8.0
    cut = K.attn_kept(q, k, lse, heads, scale, 1e-3, budget, 64, 0, heads)
    n = cut.cols.numel()
    assert n < int(cut.total) == int(full.total) and int(cut.row_ptr[-1]) == n
    assert torch.equal(cut.cols, full.cols[:n]) and torch.equal(cut.vals, full.vals[:n])
    with pytest.raises(RuntimeError):
        budget.sync_check()
    same = K.SparseRows(cut.row_ptr, full.cols[:n].contiguous(), full.vals[:n].contiguous(), cut.shape)
    for a, b in zip(K.attn_kept_bwd(g, q, k, v, [cut], heads, scale), K.attn_kept_bwd(g, q, k, v, [same], heads, scale)):
        assert torch.equal(a, b) and bool(torch.isfinite(a).all())


def test_what_is_refused(K):
    B, S, heads, hd = 1, 64, 2, 64
    q, k, v, g = tensors(B, S, heads, hd)
    out, lse = K.attn_fwd(q, k, v, heads, 0.1)
    for thr in (0.0, -1.0, 1.0, float("nan")):
        assert K.attn_kept_entries(K.KeptBudget(), thr, S, hd) == 0
        with pytest.raises(NotImplementedError):
            K.attn_kept(q, k, lse, heads, 0.1, thr, None, 8, 0, heads)
    with pytest.raises(ValueError):
        K.attn_kept(q, k, lse, heads, 0.1, 0.1, None, 8, 1, heads)       # a matrix past the last
    kept = K.attn_kept(q, k, lse, heads, 0.1, 0.1, None, 8, 0, heads)
    with pytest.raises(ValueError):
        K.attn_kept_bwd(g, q, k, v, [kept, kept], heads, 0.1)
    budget = K.KeptBudget()
    budget.observe(S * S * 0.01, S)
    assert K.attn_kept_entries(budget, 0.1, S, hd) == 32
    assert not any((K.attn_kept_entries(budget, 0.1, S, 32), K.attn_kept_entries(budget, 0.1, 60, hd), K.attn_kept_entries(budget, 0.1, 8192, hd)))


@pytest.mark.parametrize("heads,S,group_bytes", [(8, 256, 128 << 20), (4, 224, 3 * 4 * 224 * 32)])
def test_layer_step_without_score_matrices(hyc, K, heads, S, group_bytes):
    """a calibrated layer's step and the same step with the score matrices written out: output and gradients agree as two
    evaluations in bf16 do (the scores of the latter are rounded to bf16, 2^-9 of up to 8, before the exponential)"""
    import importlib
    DL = importlib.import_module("hyc-lora_amd.decoder_layer")
    cfg = DL.LayerConfig(hidden=512, heads=heads, head_dim=512 // heads, intermediate=1024, lora_r=8, act_bits=8, linear_bits=8,
                         act_group=64, attn_group_bytes=group_bytes)
    torch.manual_seed(3)
    layer = DL.DecoderLayer(cfg)
    x = torch.randn(2, S, 512, device="cuda").bfloat16().requires_grad_(True)
    g = torch.randn(2, S, 512, device="cuda").bfloat16()
    params = [x] + list(layer.parameters())
    calls = []
    inner = K.attn_kept
    def step():
        y = layer(x)
        return [y.detach()] + list(torch.autograd.grad(y, params, g, allow_unused=True))
    with torch.no_grad():
        layer(x), layer(x)
    plain = step()                                  # the first calibrated step measures how much is kept
    try:
        K.attn_kept = lambda *a: calls.append(a[-2:]) or inner(*a)
        kept = step()
    finally:
        K.attn_kept = inner
    assert sum(n for _, n in calls) == 2 * heads and len(calls) == (1 if group_bytes == 128 << 20 else 3)
    for a, b in zip(kept, plain):
        if a is not None:
            close(a, b, 0.03)
