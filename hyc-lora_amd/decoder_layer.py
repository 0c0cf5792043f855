"""One LLaMA-shaped decoder layer with a 4-bit NF4 frozen base, LoRA on all seven projections and every saved
activation compressed: the harness for the full-layer configuration (peak activation memory and step time).

What the reference assembles by swapping modules inside models/modeling_llama.py (attention :382-484, MLP
:263-295) with peft LoRA around a bitsandbytes 4-bit base (bitsandbytes_fix/_function.py:509-540) is built here
directly from this package's operators, with the savings a hand-assembled layer allows:

* q/k/v (and gate/up) LoRA-A inputs are the same tensor: it is compressed once, not once per projection;
* the attention probabilities are kept once (the reference keeps them in the softmax module and again in the
  p @ v wrapper, efficient_gemm.py:222);
* the frozen base saves nothing (as in the reference): W is dequantised again in the backward.

Composite of one LoRA projection (peft `Linear.forward` around the swapped modules):
    y  = x @ W^T + s * (x @ A^T) @ B^T          h = x @ A^T is kept exactly ([M, r])
    dX = dY @ W + (s * dY @ B) @ A
    dB = s * dY^T @ h
    dA = (s * dY @ B)^T @ x_hat                 the only consumer of the compressed x (efficient_linear.py:56-67)
"""
import functools
import math
from dataclasses import dataclass

import torch

from . import kernels as K
from .operators._calibration import CompressionSite, running_mean
from .operators.compress_function import get_statistics_softmax
from .operators.efficient_hadamard import EfficientMemoryGatedAct, _row_view
from .operators.efficient_rmsnorm import EfficientMemoryRMSNorm

BF16 = torch.bfloat16


@dataclass
class LayerConfig:
    hidden: int = 4096
    heads: int = 32
    head_dim: int = 128
    intermediate: int = 11008
    rope_theta: float = 10000.0
    rms_eps: float = 1e-5
    lora_r: int = 16
    lora_alpha: float = 32.0
    outlier_ratio: float = 0.01      # fraction of channels kept in bf16 at every compressed site
    softmax_ratio: float = 0.01      # fraction of attention probabilities kept
    linear_bits: int = 2             # LoRA-A inputs
    linear_group: int = 64
    act_bits: int = 4                # norm inputs, q / k / v, gate / act(gate) / up
    act_group: int = 128
    scale_rule: str = "absmax"       # how a (token, group) scale is formed, see kernels.ChannelPlan
    compress: bool = True            # False: the same functions keep their activations in bf16 (formula check)
    attention: str = "eager"         # "eager": scores, softmax, p @ v with the kept probabilities (the path the
                                     # reference wires into its models); "flash": fused attention kernels with
                                     # q, k, v and the output saved as codes (operators/efficient_flashattention.py)
    attn_group_bytes: int = 128 << 20  # attention is walked in groups of [S, S] score matrices of at most this size


# ---- frozen base + LoRA -----------------------------------------------------------------------------------
class LoRAProjections(torch.nn.Module):
    """n projections of one input: frozen NF4 base W_i [out_i, in] plus trainable A_i [r, in], B_i [out_i, r]"""

    def __init__(self, in_features, out_features, cfg: LayerConfig, device):
        super().__init__()
        gen = torch.Generator(device="cpu").manual_seed(in_features * 31 + sum(out_features))
        self.in_features, self.out_features = in_features, list(out_features)
        self.scaling = cfg.lora_alpha / cfg.lora_r
        self.cfg = cfg
        self.lora_A = torch.nn.ParameterList()
        self.lora_B = torch.nn.ParameterList()
        weights = []
        for out in self.out_features:
            weights.append((0.02 * torch.randn(out, in_features, generator=gen)).to(BF16).to(device))
            a = torch.empty(cfg.lora_r, in_features)
            torch.nn.init.kaiming_uniform_(a, a=math.sqrt(5), generator=gen)
            self.lora_A.append(torch.nn.Parameter(a.to(BF16).to(device)))
            # peft starts B at zero; a small random B keeps every gradient of the harness non-trivial
            self.lora_B.append(torch.nn.Parameter((0.02 * torch.randn(out, cfg.lora_r, generator=gen)).to(BF16).to(device)))
        # the frozen weights of the group live as one [sum(out), in] NF4 matrix: one dequantisation and one base GEMM
        # per forward (a three times wider GEMM runs 15-25 % faster than three); base[i] are views of projection i
        self.base_all = K.nf4_quantize(torch.cat(weights, dim=0))
        del weights
        self.base, row = [], 0
        for out in self.out_features:
            lo, hi = row * in_features, (row + out) * in_features
            self.base.append(K.NF4Weight(self.base_all.packed[lo // 2:hi // 2], self.base_all.absmax[lo // 64:hi // 64],
                                         (out, in_features)))
            row += out
        self.site = CompressionSite(cfg.outlier_ratio, 1.0, cfg.linear_bits, "per-token", 0, "hyc", cfg.linear_group,
                                    cfg.scale_rule)
        self.iteration = 0
        self.record = None

    @property
    def room(self):
        """columns for the group's rank columns behind its gradients (of the factors as they are now: a rank may be changed)"""
        return K.lora_room(len(self.out_features), self.lora_A[0].shape[0])

    def forward(self, x):
        x2 = x.reshape(-1, self.in_features)
        plan = self.site.channel_plan(x2, self.iteration) if self.cfg.compress else None
        self.iteration += 1
        outs = _LoRAProjectionsFunc.apply(x, self, plan, *self.lora_A, *self.lora_B)
        return outs if len(self.out_features) > 1 else outs[0]


@functools.lru_cache(maxsize=1024)
def _cut_columns(M, N):
    """columns at which _product cuts an [M, N] result in two, 0 to leave it whole.  The library's kernels are chosen for
    256-wide tiles here, and where they do not come out even it takes ones that run at down to half the rate.  A cut behind the
    first 8192 columns (4096 of up to 8192) costs nothing where the two parts take no more rounds of 256 tiles over the 256
    CUs than the whole does, and gains where the first part fills its rounds and the rest is short, or where the width is a
    multiple of 256 that no 192- or 224-wide tile divides.  Measured at 22 widths from 4608 to 37888 and 25 token counts from
    1024 to 16384, both with and without accumulation: 328 products that this rule cuts take 1.23 times as long whole on
    average, and one of them 0.93 times (the next 0.97).  In us, whole -> cut: N = 22016, K = 4096 at 1536 / 2048 / 3093 /
    4096 tokens 288 -> 213, 401 -> 253, 536 -> 421, 625 -> 497; N = 11008, K = 4160: 130 -> 121, 260 -> 142, 328 -> 228,
    404 -> 266; N = 5632, K = 2112 at 3093 / 4096: 80 -> 74, 94 -> 79.  Left whole for the rounds a cut adds: N = 22016 at
    2560 and 5120 tokens 326 (361 cut) and 736 (860), N = 11008 at 2560 160 (189), N = 5632 at 2048 52 (54); for its width:
    N = 13824, K = 5120 at 2048 tokens 207 (212), N = 27648, K = 4096 the same 332 (443)."""
    if N % 256 or N % 4096 == 0 or N <= 4096 or M * N <= 256 * 256 * 256:
        return 0
    cut = 8192 if N > 8192 else 4096
    rest, row_tiles = N - cut, -(-M // 256)
    rounds = lambda columns: -(-row_tiles * (columns // 256) // 256)
    first = row_tiles * (cut // 256)                                # tiles of the first part
    if rounds(cut) > 4 or rounds(cut) + rounds(rest) > rounds(N):
        return 0
    even = first % 256 == 0
    if even and 2 * rest <= cut:
        return cut
    filled = even or (rounds(cut) <= 2 and 4 * first >= 3 * 256 * rounds(cut))
    return cut if filled and (N // 256) % 3 and (N // 256) % 7 else 0


@functools.lru_cache(maxsize=1024)
def _parts(M, N):
    """(column, column, row, row) ranges of an [M, N] result that accumulates, each of at most 256 tiles of 256 x 256, one per CU.

    The library's accumulating products leave wrong values now and then where a workgroup takes more than one tile: about 1000
    elements of one 128 x 128 block, off by up to 2.7 times the result's root mean square, in 6 of 500 calls at 4096 x 12288 x 4096
    (768 tiles), 2 of 250 at 4096 x 13824 x 4096, 6 of 250 at 8192 x 8192 x 4096, 3 of 250 at 8192 x 4096 x 11008; in place and out of
    place alike, and none in 11 000 calls that do not accumulate.  In these parts there was none in 214 500 calls (6 weights, 7 token
    counts from 1024 to 8192), with the same bits.  A part fills a round of the CUs, so that they take no longer; us, as the library
    takes them in one or in two (_cut_columns) -> in parts: 12288 x 4096 at 2048 / 4096 / 8192 tokens 200 -> 168, 313 -> 334,
    633 -> 643; 22016 x 4096 306 -> 329, 611 -> 607, 1285 -> 1183; 27648 x 5120 569 -> 503, 1108 -> 954, 2047 -> 1917."""
    down, across = -(-M // 256), -(-N // 256)
    best = None
    for shares in range(1, down + 1):
        rows = -(-down // shares)
        columns = min(256 // rows, across) if rows <= 256 else 0
        if columns:
            count = -(-down // rows) * -(-across // columns)
            if best is None or count < best[0]:
                best = count, 256 * rows, 256 * columns
            if count == 1 or columns == across:
                break
    return tuple((c, min(c + best[2], N), r, min(r + best[1], M)) for c in range(0, N, best[2]) for r in range(0, M, best[1])) if best else ()


def _product(out, a, b, accumulate=False):
    """out [M, N] (+)= a @ b^T, both operands contiguous along the reduction, in one product or more (_cut_columns, _parts); over few
    rows by the package's own (kernels.few_rows)"""
    M, N = out.shape
    if accumulate:
        for c0, c1, r0, r1 in _parts(M, N):
            out[r0:r1, c0:c1].addmm_(a[r0:r1], b[c0:c1].t())
        return
    if K.few_rows(out, a, b):
        return
    cut = _cut_columns(M, N)
    for lo, hi in (((0, cut), (cut, N)) if cut else ((0, N),)):
        torch.mm(a, b[lo:hi].t(), out=out[:, lo:hi])


def _room_behind(rows, tensors, total, room):
    """`rows` if it is the [M, total + room] buffer whose first columns `tensors` are, side by side, else None"""
    if not isinstance(rows, torch.Tensor) or rows.dtype != BF16 or rows.dim() != 2 or not rows.is_contiguous():
        return None
    if rows.shape[1] != total + room or any(t.dtype != BF16 or t.numel() != rows.shape[0] * t.shape[-1] for t in tensors):
        return None
    at = rows.data_ptr()
    for t in tensors:
        t2 = t.flatten(0, -2) if t.dim() > 2 else t
        if t2.data_ptr() != at or t2.stride(1) != 1 or (t2.shape[0] > 1 and t2.stride(0) != total + room):
            return None
        at += 2 * t.shape[-1]
    return rows


def _kernel_rows(t):
    """[..., H] -> the [M, H] rows the kernels read as they lie (16-byte aligned, evenly spaced by a multiple of 8 elements, none
    on top of another), copied where they do not: a gradient broadcast over the tokens, an odd slice, a view at an odd offset"""
    t = _row_view(t)
    if t.data_ptr() % 16 or (t.shape[0] > 1 and (t.stride(0) < t.shape[1] or t.stride(0) % 8)):
        t = t.clone(memory_format=torch.contiguous_format)
    return t


class _LoRAProjectionsFunc(torch.autograd.Function):
    """A group is one product each way: forward y = s h B^T (h = x A^T), onto which the base product accumulates in its epilogue (in
    parts, see _parts; over few tokens both in one launch from the codes, kernels.few_rows_base); backward dX = [dY | s dY B] [W^T |
    A^T]^T with the rank-r terms as further columns of the reduction (kernels.lora_down / lora_up / lora_up_bwd / lora_weight_t)."""

    @staticmethod
    def forward(ctx, x, mod, plan, *ab):
        n, cfg = len(mod.out_features), mod.cfg
        A, B = ab[:n], ab[n:]
        if mod.record is None and (plan is not None) == cfg.compress:
            outs, r, M = tuple(mod.out_features), A[0].shape[0], x.numel() // mod.in_features
            if K._lora_kernels_cover(M, n, r, mod.in_features, outs):
                done = K.native.lora_forward(x, A, B, mod.scaling, outs, mod.base_all.packed, mod.base_all.absmax,
                                             _parts(M, sum(outs)), plan, cfg.linear_bits, cfg.linear_group)
                if done is not None:
                    ys, ctx.h, ctx.saved_x = done
                    if not cfg.compress:
                        ctx.saved_x = _kernel_rows(x).contiguous()
                    ctx.mod = mod
                    ctx.save_for_backward(*ab)
                    return ys
        x2 = _kernel_rows(x)
        h = K.lora_down(x2, A)
        y_all = K.few_rows_base(x2, mod.base_all, h, B, mod.scaling, mod.out_features)
        if y_all is None:
            y_all = K.lora_up(h, B, mod.scaling, mod.out_features)
            _product(y_all, x2, K.nf4_dequantize(mod.base_all), accumulate=True)
        outs, row = [], 0
        for out in mod.out_features:                            # column slices: no copies, consumers take the pitch
            outs.append(y_all[:, row:row + out].unflatten(0, x.shape[:-1]))
            row += out
        ctx.saved_x = K.compress_channel(x2, plan, cfg.linear_bits, cfg.linear_group) if cfg.compress else x2.contiguous()
        if mod.record is not None:
            mod.record["x"], mod.record["saved"] = x2.detach().clone(), ctx.saved_x
        ctx.mod, ctx.h = mod, h
        ctx.save_for_backward(*ab)
        return tuple(outs)

    @staticmethod
    def backward(ctx, *gs):
        mod = ctx.mod
        n = len(mod.out_features)
        A, B = ctx.saved_tensors[:n], ctx.saved_tensors[n:]
        r, total = A[0].shape[0], sum(mod.out_features)
        if torch.is_grad_enabled():                             # create_graph: products that leave one
            return _LoRAProjectionsFunc._backward_with_graph(ctx, A, B, gs)
        room = K.lora_room(n, r)
        rows = _room_behind(getattr(gs[0], "_hyc_rows", None), gs, total, room)
        if not K.gradw_staged_by_default(32, mod.in_features):
            M, outs = ctx.h.shape[0], tuple(mod.out_features)
            if K._lora_kernels_cover(M, n, r, mod.in_features, outs):
                done = K.native.lora_backward(gs, A, B, ctx.h, mod.scaling, outs, room, rows, mod.base_all.packed, mod.base_all.absmax,
                                              ctx.saved_x, _cut_columns(M, mod.in_features))
                if done is not None:
                    ctx.h = ctx.saved_x = None
                    return done[:1] + (None, None) + done[1:]
        ext, dh, dB = K.lora_up_bwd([_kernel_rows(g.to(BF16)) for g in gs], B, ctx.h, mod.scaling, room, rows)
        dA = _LoRAProjectionsFunc._grad_A(ctx, dh, A)
        dx = torch.empty((ext.shape[0], mod.in_features), dtype=BF16, device=ext.device)
        _product(dx, ext, K.lora_weight_t(mod.base_all, A, mod.out_features, room))
        ctx.h = ctx.saved_x = None
        return (dx.reshape(gs[0].shape[:-1] + (mod.in_features,)), None, None) + tuple(dA) + tuple(dB)

    @staticmethod
    def _grad_A(ctx, dh, A):
        """dA_i = dh_i^T @ x_hat: the projections of a group read the same saved activation, so their dh go through the
        weight-gradient kernel side by side, up to 128 rows a call where its sums keep the order they have with up to 32
        (kernels.gradw_rows_per_call; otherwise they lose precision): one launch, and one that adds up the partial results, for the
        whole group.  Two or three calls of up to 32 rows -> one, us, codes of 2 | 4 | 8 bits | dense:
        48 rows of 157 x 2048 13.9 -> 6.9 | 13.9 -> 7.0 | 11.6 -> 7.0 | 12.9 -> 9.7, 1000 x 1024 17.7 -> 8.9 | 17.7 -> 8.9 |
        16.0 -> 8.9 | 14.3 -> 10.6, 157 x 11008 14.1 -> 7.2 | 14.1 -> 7.2 | 11.9 -> 7.2 | 14.7 -> 11.9; 96 rows of 157 x 2048
        19.4 -> 7.0 | 19.5 -> 7.1 | 19.6 -> 7.1 | 19.8 -> 10.6.  From about 2000 tokens on codes take 32 rows a call (dense sources
        keep their order, 48 and 96 rows of 4096 x 4096 28.1 -> 27.2 and 45.9 -> 32.3): one call would be faster there too, 48
        rows of 2048 x 4096 20.1 -> 13.8, 4096 x 4096 23.2 -> 14.6, 4096 x 11008 38.1 -> 26.0 (2 bits)."""
        r, dA = A[0].shape[0], []
        per_call = K.gradw_rows_per_call(dh.shape[0], dh.shape[1], r, ctx.saved_x)
        for c0 in range(0, dh.shape[1], per_call):
            block = K.gradw_gemm(dh[:, c0:c0 + per_call], ctx.saved_x, out_dtype=A[0].dtype)
            dA.extend(block[j:j + r] for j in range(0, block.shape[0], r))
        return dA

    @staticmethod
    def _backward_with_graph(ctx, A, B, gs):
        """the same gradients through torch's own products, so that dx and dB can be differentiated again with respect to the
        gradients and the factors (dA comes from the compressed input by a kernel and is a constant there)"""
        mod, s, r = ctx.mod, ctx.mod.scaling, A[0].shape[0]
        gs2 = [g.reshape(-1, o).to(BF16) for g, o in zip(gs, mod.out_features)]
        dhs = [s * (g @ b) for g, b in zip(gs2, B)]
        dB = [s * (g.t() @ ctx.h[:, i * r:(i + 1) * r]) for i, g in enumerate(gs2)]
        dh = torch.cat(dhs, dim=1)
        dA = _LoRAProjectionsFunc._grad_A(ctx, dh.detach(), A)
        dx = dh @ torch.cat(list(A), dim=0) + torch.cat(gs2, dim=1) @ K.nf4_dequantize(mod.base_all)
        ctx.h = ctx.saved_x = None
        return (dx.reshape(gs[0].shape[:-1] + (mod.in_features,)), None, None) + tuple(dA) + tuple(dB)


# ---- attention -----------------------------------------------------------------------------------------------
def rope_tables(S, head_dim, theta, device):
    inv = 1.0 / (theta ** (torch.arange(0, head_dim, 2, dtype=torch.float32, device=device) / head_dim))
    freqs = torch.outer(torch.arange(S, dtype=torch.float32, device=device), inv)
    emb = torch.cat((freqs, freqs), dim=-1)
    return emb.cos().to(BF16), emb.sin().to(BF16)


class CompressedAttention(torch.nn.Module):
    """RoPE, softmax(q @ k^T / sqrt(hd) + causal mask) @ v on the [B, S, H] projections, with q, k (after RoPE) and v
    saved as codes in the [B*S, nh*hd] layout and the probabilities saved once as the entries above a calibrated
    threshold.  Composition of apply_rotary_pos_emb and the reference's gemm1, softmax and gemm2 modules
    (models/modeling_llama.py:423-462, operators/efficient_gemm.py, operators/efficient_softmax.py)."""

    # a number of columns: where one kernel writes the gradients of q, k and v, they lie side by side in one matrix with that many
    # free columns behind them, which is handed on as `_hyc_rows` of the three (see _LoRAProjectionsFunc); None: three
    # contiguous tensors
    grad_room = None

    def __init__(self, cfg: LayerConfig):
        super().__init__()
        if cfg.attention not in ("eager", "flash"):
            raise ValueError("attention must be 'eager' or 'flash', got %r" % (cfg.attention,))
        self.cfg = cfg
        mk = lambda: CompressionSite(cfg.outlier_ratio, 1.0, cfg.act_bits, "per-token", 0, "hyc", cfg.act_group,
                                     cfg.scale_rule)
        self.site_q, self.site_k, self.site_v, self.site_o = mk(), mk(), mk(), mk()
        self.iteration = 0
        self.static_value = None          # probability threshold, as in EfficientMemorySoftmax
        self.record = None

    def forward(self, q, k, v, cos, sin, grad_room=None):
        grad_room = self.grad_room if grad_room is None else grad_room
        func = _FlashAttentionFunc if self.cfg.attention == "flash" else _AttentionFunc
        return func.apply(q, k, v, cos, sin, self, grad_room)


def _frozen_plans(sites, iteration):
    """the plans of calibrated sites, None while one of them still looks at what it is given"""
    if iteration < 2 or any(site.plan is None for site in sites):
        return None
    return tuple(site.plan for site in sites)


def _compress_sites(sites, tensors, iteration, cfg):
    out = []
    for site, t in zip(sites, tensors):
        t = t.reshape(-1, t.shape[-1])
        out.append(K.compress_channel(t, site.channel_plan(t, iteration), cfg.act_bits, cfg.act_group))
    return out


def _matrices_per_group(total, s, budget_bytes):
    """[S, S] bf16 score matrices per group: within the budget, and the groups of equal size"""
    most = max(1, min(total, budget_bytes // (2 * s * s)))
    groups = -(-total // most)
    return -(-total // groups)


class _AttentionFunc(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, cos, sin, mod, grad_room):
        cfg = mod.cfg
        b, s, H = q.shape
        nh, hd = cfg.heads, cfg.head_dim
        scale = 1.0 / math.sqrt(hd)
        ctx.rows = _AttentionFunc._without_matrices(q, k, v, mod, grad_room)
        if ctx.rows:
            return _AttentionFunc._forward_kept(ctx, q, k, v, cos, sin, mod, grad_room)
        # one pass per tensor: rotate, and write both the head-major copy the batched GEMMs need and the rows that
        # are compressed
        qh, q_rows = K.rope_to_heads(q, nh, cos, sin, want_rows=True)
        kh, k_rows = K.rope_to_heads(k, nh, cos, sin, want_rows=True)
        v_rows = v                                                # possibly a column slice of the fused projection
        vh = K.rope_to_heads(v_rows, nh)
        # The [S, S] score matrices are processed in groups that bound the transient tensors (they stay in
        # the last-level cache and the peak memory no longer grows with B * heads): per group one library GEMM for
        # scores = (q @ k^T) / sqrt(hd), the softmax kernel with the causal mask built in (the masked half is never
        # read; the probabilities overwrite the scores), one GEMM for p @ v.
        q3, k3, v3 = qh.view(b * nh, s, hd), kh.view(b * nh, s, hd), vh.view(b * nh, s, hd)
        group = _matrices_per_group(b * nh, s, cfg.attn_group_bytes)
        it = mod.iteration
        calibrating = cfg.compress and it < 2
        if calibrating:
            group = b * nh                 # the threshold is a quantile over batch element 0: all of it is needed
        zero = q.new_zeros(1)
        out3 = torch.empty_like(q3)
        kept, p_all = [], None
        for c0 in range(0, b * nh, group):
            c1 = min(c0 + group, b * nh)
            scores = torch.baddbmm(zero, q3[c0:c1], k3[c0:c1].transpose(1, 2), beta=0.0, alpha=scale)
            if not cfg.compress:
                p, _ = K.softmax_fwd(scores, causal_period=s, inplace=True)
                kept.append(p)                                     # kept whole, in bf16
            elif not calibrating:
                p, sp = K.softmax_fwd(scores, K.threshold_value(mod.static_value), causal_period=s, inplace=True,
                                      budget=K.kept_budget(mod.static_value))
                kept.append(sp)
            else:
                p, _ = K.softmax_fwd(scores, causal_period=s, inplace=True)
                thr = get_statistics_softmax(p.view(b, nh, s, s), it, cfg.softmax_ratio)
                mod.static_value = running_mean(mod.static_value, thr, it)
                kept.append(K.softmax_sparsify(p, K.threshold_value(thr)))
            del scores
            torch.bmm(p, v3[c0:c1], out=out3[c0:c1])
            if mod.record is not None:
                p_all = p if p_all is None else torch.cat([p_all, p])
            del p
        out = K.rope_from_heads(out3.view(b, nh, s, hd))            # [B, S, H]
        del qh, kh, vh, q3, k3, v3, out3
        rows = [t.reshape(b * s, H) for t in (q_rows, k_rows, v_rows)]      # views (v keeps its pitch)
        if cfg.compress:
            saved = []
            for site, r in zip((mod.site_q, mod.site_k, mod.site_v), rows):
                plan = site.channel_plan(r, it)
                saved.append(K.compress_channel(r, plan, cfg.act_bits, cfg.act_group))
        else:
            saved = [r.contiguous() for r in rows]
        mod.iteration += 1
        if mod.record is not None:
            mod.record.update(q=rows[0].detach().clone(), k=rows[1].detach().clone(), v=rows[2].detach().clone(),
                              p=p_all.view(b, nh, s, s), saved=saved, sparse=list(kept))
        ctx.saved, ctx.kept, ctx.group, ctx.geom, ctx.compress = saved, kept, group, (b, nh, s, hd), cfg.compress
        ctx.save_for_backward(cos, sin)
        return out

    @staticmethod
    def _without_matrices(q, k, v, mod, grad_room):
        """whether no score matrix is formed: a calibrated site that kernels.attn_kept_covers, whose probabilities nobody records and
        whose rows the attention kernels read as they lie.  Decided by the configuration, the calibrated threshold and the call alone,
        so that a run, its repetition and one resumed from its state take the same form at every step."""
        cfg = mod.cfg
        if not cfg.compress or mod.iteration < 2 or mod.record is not None or q.dim() != 3 or v.data_ptr() % 16 or v.shape != q.shape:
            return False
        b, s, H = q.shape
        pitch = H if grad_room is None else 3 * H + grad_room
        return (b > 0 and v.stride(2) == 1 and v.stride(1) % 8 == 0
                and K.attn_supported(cfg.head_dim, s, max(v.stride(1), pitch), b * cfg.heads)
                and K.attn_kept_covers(K.threshold_value(mod.static_value), s, cfg.head_dim, cfg.softmax_ratio))

    @staticmethod
    def _forward_kept(ctx, q, k, v, cos, sin, mod, grad_room):
        cfg = mod.cfg
        b, s, H = q.shape
        nh = cfg.heads
        scale = 1.0 / math.sqrt(cfg.head_dim)
        sites = (mod.site_q, mod.site_k, mod.site_v)
        done = K.native.rope_attn_fwd(q, k, v, nh, cos, sin, scale, True, _frozen_plans(sites, mod.iteration), cfg.act_bits, cfg.act_group)
        if done is None:
            q_rows, k_rows = K.rope_rows(q, nh, cos, sin), K.rope_rows(k, nh, cos, sin)
            done = (q_rows, k_rows) + K.attn_fwd(q_rows, k_rows, v, nh, scale, round_scores=True) + (None,)
        q_rows, k_rows, out, lse, saved = done
        thr, budget = K.threshold_value(mod.static_value), K.kept_budget(mod.static_value)
        cap = K.attn_kept_entries(budget, thr, s, cfg.head_dim) or K.slab_room(cfg.softmax_ratio * s, s)
        # (the slab of kept entries is what grows with the number of matrices here)
        group = max(1, min(b * nh, cfg.attn_group_bytes // (4 * s * cap)))
        ctx.kept = [K.attn_kept(q_rows, k_rows, lse, nh, scale, thr, budget, cap, c0, min(group, b * nh - c0))
                    for c0 in range(0, b * nh, group)]
        ctx.saved = saved or _compress_sites(sites, (q_rows, k_rows, v), mod.iteration, cfg)
        mod.iteration += 1
        ctx.geom, ctx.grad_room = (b, nh, s, cfg.head_dim), grad_room
        ctx.save_for_backward(cos, sin)
        return out

    @staticmethod
    def backward(ctx, g):
        b, nh, s, hd = ctx.geom
        cos, sin = ctx.saved_tensors
        if ctx.rows:
            grads = K.native.attn_kept_bwd(g, *ctx.saved, ctx.kept, nh, cos, sin, 1.0 / math.sqrt(hd), ctx.grad_room)
            if grads is None:
                qq, kk, vv = (K.decompress_channel(c).view(b, s, nh * hd) for c in ctx.saved)
                grads = K.attn_kept_bwd(g.to(BF16).contiguous(), qq, kk, vv, ctx.kept, nh, 1.0 / math.sqrt(hd), cos, sin, room=ctx.grad_room)
            ctx.saved = ctx.kept = None
            if ctx.grad_room is not None:
                for t in grads[:3]:
                    t._hyc_rows = grads[3]
            return grads[:3] + (None,) * 4
        restore = (lambda c: K.decompress_channel(c)) if ctx.compress else (lambda c: c)
        to_heads = lambda rows: K.rope_to_heads(rows.view(b, s, nh * hd), nh).view(b * nh, s, hd)
        gh = K.rope_to_heads(g.to(BF16).contiguous(), nh).view(b * nh, s, hd)
        v = to_heads(restore(ctx.saved[2]))
        kk = to_heads(restore(ctx.saved[1]))
        qq = to_heads(restore(ctx.saved[0]))
        dq, dk, dv = torch.empty_like(qq), torch.empty_like(qq), torch.empty_like(qq)
        scale = 1.0 / math.sqrt(hd)
        zero = gh.new_zeros(1)                                     # ignored (beta = 0), only has to broadcast
        for i, c0 in enumerate(range(0, b * nh, ctx.group)):
            c1 = min(c0 + ctx.group, b * nh)
            item = ctx.kept[i]
            p = K.softmax_dense(item) if ctx.compress else item
            torch.bmm(p.transpose(1, 2), gh[c0:c1], out=dv[c0:c1])
            dp = torch.bmm(gh[c0:c1], v[c0:c1].transpose(1, 2))
            if ctx.compress:
                del p
                ds = K.softmax_bwd(dp, item, inplace=True)
            else:
                ds = torch._softmax_backward_data(dp, p, -1, BF16)
                del p
            del dp
            torch.baddbmm(zero, ds, kk[c0:c1], beta=0.0, alpha=scale, out=dq[c0:c1])
            torch.baddbmm(zero, ds.transpose(1, 2), qq[c0:c1], beta=0.0, alpha=scale, out=dk[c0:c1])
            del ds
            ctx.kept[i] = None
        del v, kk, qq, gh
        ctx.saved = ctx.kept = None
        dq = K.rope_from_heads(dq.view(b, nh, s, hd), cos, sin)
        dk = K.rope_from_heads(dk.view(b, nh, s, hd), cos, sin)
        dv = K.rope_from_heads(dv.view(b, nh, s, hd))
        return dq, dk, dv, None, None, None, None


class _FlashAttentionFunc(torch.autograd.Function):
    """The design of the reference's flash-attention operator (operators/efficient_flashattention.py:10-135): a fused
    attention kernel (hyc_attn_fwd; the library's for head sizes other than 64 and 128) runs the forward, what is kept is
    q, k (after RoPE), v and the attention output as codes plus the fp32 log-sum-exp of every row, and the fused backward runs on the restored
    tensors.  No [S, S] matrix exists at any time.  The backward kernel rebuilds the probabilities from the restored
    q and k with the exact log-sum-exp, and takes its row term sum(dO * O) from the restored output."""

    @staticmethod
    def forward(ctx, q, k, v, cos, sin, mod, grad_room):
        cfg = mod.cfg
        b, s, H = q.shape
        nh, hd = cfg.heads, cfg.head_dim
        scale = 1.0 / math.sqrt(hd)
        pitch = H if grad_room is None else 3 * H + grad_room       # of the gradients
        ctx.rows = K.attn_supported(hd, s, max(v.stride(1), pitch), b * nh)
        sites, it = (mod.site_q, mod.site_k, mod.site_v, mod.site_o), mod.iteration
        seed = offset = saved = None
        if ctx.rows:                                                # the kernels read and write the rows as they are
            plans = _frozen_plans(sites, it) if cfg.compress else None
            done = K.native.rope_attn_fwd(q, k, v, nh, cos, sin, scale, False, plans, cfg.act_bits, cfg.act_group)
            if done is None:
                q_rows, k_rows = K.rope_rows(q, nh, cos, sin), K.rope_rows(k, nh, cos, sin)
                done = (q_rows, k_rows) + K.attn_fwd(q_rows, k_rows, v, nh, scale) + (None,)
            q_rows, k_rows, out, lse, saved = done
            ctx.grad_room = grad_room
        else:
            qh, q_rows = K.rope_to_heads(q, nh, cos, sin, want_rows=True)
            kh, k_rows = K.rope_to_heads(k, nh, cos, sin, want_rows=True)
            vh = K.rope_to_heads(v, nh)
            out_h, lse, _, _, _, _, seed, offset, _ = torch.ops.aten._scaled_dot_product_flash_attention(
                qh, kh, vh, 0.0, True, False, scale=scale)
            del qh, kh, vh
            out = K.rope_from_heads(out_h)                          # [B, S, H]
            del out_h
        rows = [t.reshape(b * s, H) for t in (q_rows, k_rows, v, out)]
        if cfg.compress:
            saved = saved or _compress_sites(sites, rows, it, cfg)
        else:
            saved = [r.contiguous() for r in rows]
        mod.iteration += 1
        if mod.record is not None:
            mod.record.update(q=rows[0].detach().clone(), k=rows[1].detach().clone(), v=rows[2].detach().clone(),
                              o=rows[3].detach().clone(), saved=saved, lse=lse)
        ctx.saved, ctx.geom, ctx.compress, ctx.rng = saved, (b, nh, s, hd), cfg.compress, (seed, offset)
        ctx.save_for_backward(cos, sin, lse)
        return out

    @staticmethod
    def backward(ctx, g):
        b, nh, s, hd = ctx.geom
        cos, sin, lse = ctx.saved_tensors
        restore = (lambda c: K.decompress_channel(c)) if ctx.compress else (lambda c: c)
        if ctx.rows:
            saved, ctx.saved = list(ctx.saved), None                # (emptied by the call: the gradients take the codes' room)
            grads = K.native.attn_bwd(g, saved, lse, nh, cos, sin, 1.0 / math.sqrt(hd), ctx.grad_room) if ctx.compress else None
            if grads is None:
                qq, kk, vv, oo = (restore(c).view(b, s, nh * hd) for c in saved)
                saved.clear()
                grads = K.attn_bwd(g.to(BF16).contiguous(), qq, kk, vv, oo, lse, nh, 1.0 / math.sqrt(hd), cos, sin, room=ctx.grad_room)
            if ctx.grad_room is not None:
                for t in grads[:3]:
                    t._hyc_rows = grads[3]
            return grads[:3] + (None,) * 4
        to_heads = lambda rows: K.rope_to_heads(rows.view(b, s, nh * hd), nh)
        gh = K.rope_to_heads(g.to(BF16).contiguous(), nh)
        qq, kk, vv, oo = (to_heads(restore(c)) for c in ctx.saved)
        ctx.saved = None
        dq, dk, dv = torch.ops.aten._scaled_dot_product_flash_attention_backward(
            gh, qq, kk, vv, oo, lse, None, None, s, s, 0.0, True, ctx.rng[0], ctx.rng[1], scale=1.0 / math.sqrt(hd))
        del gh, qq, kk, vv, oo
        dq = K.rope_from_heads(dq.contiguous(), cos, sin)
        dk = K.rope_from_heads(dk.contiguous(), cos, sin)
        dv = K.rope_from_heads(dv.contiguous())
        return dq, dk, dv, None, None, None, None


# ---- the layer --------------------------------------------------------------------------------------------------
class _PlainRMSNorm(torch.nn.Module):
    def __init__(self, hidden, eps, device):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(hidden, dtype=BF16, device=device))
        self.eps = eps

    def forward(self, x):
        xf = x.float()
        return (self.weight.float() * (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps))).to(x.dtype)


class DecoderLayer(torch.nn.Module):
    def __init__(self, cfg: LayerConfig = None, device="cuda"):
        super().__init__()
        self.cfg = cfg = cfg or LayerConfig()
        H, I = cfg.hidden, cfg.intermediate
        if cfg.heads * cfg.head_dim != H:
            raise ValueError("heads * head_dim must equal hidden")
        if cfg.compress:
            norm = lambda: EfficientMemoryRMSNorm(H, eps=cfg.rms_eps, elementwise_affine=True, bias=False,
                                                  outlier_ratio=cfg.outlier_ratio, sub_outlier_ratio=1.0,
                                                  sub_outlier_bit=cfg.act_bits, sub_outlier_quantize_method="per-token",
                                                  rank=0, mode="hyc", group_size=cfg.act_group,
                                                  scale_rule=cfg.scale_rule).to(device).to(BF16)
        else:
            norm = lambda: _PlainRMSNorm(H, cfg.rms_eps, device)
        self.input_layernorm = norm()
        self.post_attention_layernorm = norm()
        self.qkv_proj = LoRAProjections(H, [H, H, H], cfg, device)
        self.o_proj = LoRAProjections(H, [H], cfg, device)
        self.gate_up_proj = LoRAProjections(H, [I, I], cfg, device)
        self.down_proj = LoRAProjections(I, [H], cfg, device)
        self.attention = CompressedAttention(cfg)
        self.act = EfficientMemoryGatedAct("silu", cfg.outlier_ratio, 1.0, cfg.act_bits, "per-token", 0,
                                           group_size=cfg.act_group, scale_rule=cfg.scale_rule) if cfg.compress else None
        # (as attributes: what the layer calls its modules with is what their hooks and replacements see)
        self.attention.grad_room = self.qkv_proj.room
        if self.act is not None:
            self.act.grad_room = self.gate_up_proj.room
        self._rope = None

    def forward(self, x):
        cfg = self.cfg
        b, s, H = x.shape
        if self._rope is None or self._rope[0].shape[0] != s:
            self._rope = rope_tables(s, cfg.head_dim, cfg.rope_theta, x.device)
        cos, sin = self._rope
        # no names for the wide intermediates: each is released as soon as its consumer has run
        x = x + self.o_proj(self.attention(*self.qkv_proj(self.input_layernorm(x)), cos, sin))
        return x + self.down_proj(self._gated(*self.gate_up_proj(self.post_attention_layernorm(x))))

    def _gated(self, gate, up):
        if self.act is not None:
            return self.act(gate, up)
        return torch.nn.functional.silu(gate) * up

    def saved_activation_bytes(self, batch, seq):
        """analytic size of what one forward keeps for the backward (the probabilities' share is data dependent:
        `softmax_ratio` of B*nh*S*S entries of 6 bytes plus row pointers; the fused attention keeps its output and
        one fp32 log-sum-exp per row instead)"""
        cfg = self.cfg
        M, H, I = batch * seq, cfg.hidden, cfg.intermediate

        def site(width, bits, group):
            k = K.num_outlier_channels(width, cfg.outlier_ratio)
            return M * (width * bits // 8 + 2 * k + 2 * (width // group))

        total = 2 * (site(H, cfg.act_bits, cfg.act_group) + 4 * M)                    # two norms: x + rstd
        total += 2 * site(H, cfg.linear_bits, cfg.linear_group)                       # qkv input (once), o input
        total += site(H, cfg.linear_bits, cfg.linear_group) + site(I, cfg.linear_bits, cfg.linear_group)  # gate/up, down
        total += 3 * site(H, cfg.act_bits, cfg.act_group)                             # q, k, v
        total += 3 * site(I, cfg.act_bits, cfg.act_group)                             # gate, act(gate), up
        total += 7 * M * cfg.lora_r * 2                                               # h = x @ A^T, exact
        rows = batch * cfg.heads * seq
        if cfg.attention == "flash":
            total += site(H, cfg.act_bits, cfg.act_group) + 4 * rows                  # attention output, log-sum-exp
        else:
            total += int(cfg.softmax_ratio * rows * seq) * 6 + 4 * (rows + 1)
        return total
