"""The kernels beside the frozen base of a LoRA projection group against the same products in fp32, at the sizes where a
tile of tokens (16, 64, 128), a block of features (256) or a factor (8 of 16 / 24 of 32 columns) is cut, and the torch form
that serves the ranks they do not cover."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def close(got, want):
    """one rounding of an fp32 sum to bf16 (8 bits of significand: at most 2^-8 of the element), plus the sums' own error (fp32,
    a few thousand terms)"""
    want = want.double()
    bound = 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max().clamp_min(1e-30)
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() / bound).max())


CASES = [(1, 64, [8], 8), (16, 256, [256, 64, 128], 16), (65, 512, [1000, 24], 24), (157, 1024, [320], 32), (130, 2816, [1024, 1024, 1024], 32),
         (300, 4096, [4096, 512], 16), (33, 256, [256, 256], 64),                   # rank 64: the torch form
         # token ranges of three tiles each (32 ranges of 192 tokens), both buffers refilled, with 24 and 32 of 32 columns
         (4200, 256, [512, 264], 24), (4200, 256, [512, 264], 32),
         # four and five tiles of 16 columns of h
         (200, 512, [64, 64], 32), (200, 512, [64, 64, 64], 24),
         # the transposed weight by four scale groups at a time (104 x 5 workgroups), the last of them cut at K = 1088
         (33, 1088, [13248], 16)]


@pytest.mark.parametrize("M,Kf,outs,r", CASES)
def test_lora_group_products(K, M, Kf, outs, r):
    n, total, room, s = len(outs), sum(outs), K.lora_room(len(outs), r), 1.5
    assert room >= n * r and room % 64 == 0
    gen = torch.Generator(device="cuda").manual_seed(M + Kf)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    A, B = [mk(r, Kf) for _ in outs], [mk(o, r) for o in outs]
    wide = mk(M, Kf + 8)
    x = wide[:, :Kf]                                                                # rows with a pitch of their own
    h = K.lora_down(x, A)
    close(h, torch.cat([x.float() @ a.float().t().contiguous() for a in A], 1))
    y = K.lora_up(h, B, s)
    close(y, torch.cat([s * (h[:, i * r:(i + 1) * r].float() @ b.float().t().contiguous()) for i, b in enumerate(B)], 1))
    gs = [mk(M, o) for o in outs]
    ext, dh, dB = K.lora_up_bwd(gs, B, h, s, room)
    close(dh, torch.cat([s * (g.float() @ b.float()) for g, b in zip(gs, B)], 1))
    for i, (g, d) in enumerate(zip(gs, dB)):
        close(d, s * (g.float().t().contiguous() @ h[:, i * r:(i + 1) * r].float()))
    assert torch.equal(ext[:, :total], torch.cat(gs, 1))                            # the copy, dh, zeros
    assert torch.equal(ext[:, total:total + n * r], dh) and not ext[:, total + n * r:].any()
    # the gradients already in front of the room: nothing is copied, the rest is the same bit for bit
    buf = torch.full_like(ext, float("nan"))
    buf[:, :total] = ext[:, :total]
    cuts = [sum(outs[:i]) for i in range(n + 1)]
    ext2, dh2, dB2 = K.lora_up_bwd([buf[:, a:b] for a, b in zip(cuts, cuts[1:])], B, h, s, room, buf)
    assert ext2 is buf and torch.equal(ext2, ext) and torch.equal(dh2, dh) and all(torch.equal(a, b) for a, b in zip(dB2, dB))
    # the transposed weight: the dequantised values and the factors themselves
    q = K.nf4_quantize(mk(total, Kf))
    wt = K.lora_weight_t(q, A, outs, room)
    assert torch.equal(wt[:, :total], K.nf4_dequantize(q).t()) and torch.equal(wt[:, total:total + n * r], torch.cat(A, 0).t())
    assert not wt[:, total + n * r:].any()


def test_gradients_side_by_side_are_recognised_only_when_they_are(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import importlib
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    buf = torch.zeros(6, 64 + 32 + 64, dtype=torch.bfloat16, device="cuda")
    a, b = buf[:, :64].unflatten(0, (2, 3)), buf[:, 64:96].unflatten(0, (2, 3))
    assert DL._room_behind(buf, [a, b], 96, 64) is buf
    assert DL._room_behind(None, [a, b], 96, 64) is None
    assert DL._room_behind(buf, [b, a], 96, 64) is None
    assert DL._room_behind(buf, [a, b.clone()], 96, 64) is None
    assert DL._room_behind(buf, [a, b], 96, 128) is None
    assert DL._room_behind(buf[:, :160].float(), [a, b], 96, 64) is None


def _group(hyc, outs=(128, 64), compress=False):
    import importlib
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    return DL, DL.LoRAProjections(256, list(outs), DL.LayerConfig(hidden=256, lora_r=16, compress=compress), "cuda")


def _gradients(mod, x, gs):
    x = x.detach().requires_grad_(True)
    return torch.autograd.grad(mod(x), [x] + list(mod.parameters()), gs)


def test_rows_that_do_not_lie_as_the_kernels_read_them(K, hyc):
    """gradients broadcast over the tokens, inputs and gradients at odd pitches and offsets: the results of their copies, bit for bit"""
    DL, mod = _group(hyc)
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    x, g = mk(1, 33, 256), [mk(1, 1, o).expand(1, 33, o) for o in (128, 64)]
    pitch, offset = mk(1, 33, 259)[..., :256], mk(33 * 256 + 1)[1:].view(1, 33, 256)
    cases = [(x, g), (x, [mk(1, 33, o + 3)[..., :o] for o in (128, 64)]), (x, [mk(33 * o + 1)[1:].view(1, 33, o) for o in (128, 64)]),
             (pitch, [mk(1, 33, o) for o in (128, 64)]), (offset, [mk(1, 33, o) for o in (128, 64)])]
    for xi, gi in cases:
        got = _gradients(mod, xi, gi)
        want = _gradients(mod, xi.clone(memory_format=torch.contiguous_format), [t.clone(memory_format=torch.contiguous_format) for t in gi])
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_factors_at_an_odd_address(K, hyc):
    """factors that are views into a flat parameter buffer at an offset the kernels do not take go through the general products"""
    DL, mod = _group(hyc)
    gen = torch.Generator(device="cuda").manual_seed(2)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    x, gs = mk(2, 17, 256), [mk(2, 17, o) for o in (128, 64)]
    want = _gradients(mod, x, gs)
    for p in mod.parameters():
        flat = torch.empty(p.numel() + 1, dtype=p.dtype, device="cuda")
        flat[1:] = p.data.flatten()
        p.data = flat[1:].view(p.shape)
    got = _gradients(mod, x, gs)
    for a, b in zip(got, want):                            # products in another order: a rounding to bf16 of h, of dh and of the result
        bound = 3 * 2.0 ** -8 * (b.float().abs() + b.float().abs().max())
        assert ((a.float() - b.float()).abs() <= bound).all()


def test_no_tokens(K):
    B = [torch.ones(64, 16, dtype=torch.bfloat16, device="cuda")]
    empty = lambda w: torch.empty(0, w, dtype=torch.bfloat16, device="cuda")
    K.lora_up_bwd([torch.ones(8, 64, dtype=torch.bfloat16, device="cuda")], B, torch.ones(8, 16, dtype=torch.bfloat16, device="cuda"), 1.0, 64)
    ext, dh, dB = K.lora_up_bwd([empty(64)], B, empty(16), 1.0, 64)
    assert ext.shape == (0, 128) and dh.shape == (0, 16) and not dB[0].any()


@pytest.mark.parametrize("r", [16, 32])
def test_no_tokens_at_the_c_entry(hyc, r):
    """dB of an empty batch is written (zero), with no other buffer given; nothing behind it is touched"""
    import ctypes
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K, lib = hyc.kernels, hyc._abi.load()
    outs = [72, 264]
    B = [torch.ones(o, r, dtype=torch.bfloat16, device="cuda") for o in outs]
    dB = [torch.full((o + 1, r), 7.0, dtype=torch.bfloat16, device="cuda") for o in outs]
    none = (ctypes.c_void_p * 2)(None, None)
    rc = lib.hyc_lora_up_bwd(none, K._i64s(outs), 0, K._i64s(outs), K._ptrs(B), None, 2, r, 1.0, None, None, 336 + 64, 64, 1, K._ptrs(dB), None,
                             K._stream())
    assert rc == 0 and all(not d[:-1].any() and (d[-1] == 7).all() for d in dB)


def test_more_tokens_than_a_range_takes_in_32(K):
    """past 32 x 32768 tokens there are more ranges, each short enough for its offsets"""
    M, r = (1 << 20) + 33, 8
    gen = torch.Generator(device="cuda").manual_seed(3)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    g, h, B = mk(M, 8), mk(M, r), [mk(8, r)]
    ext, dh, dB = K.lora_up_bwd([g], B, h, 0.5, 64)
    close(dh, 0.5 * (g.float() @ B[0].float()))
    close(dB[0], 0.5 * (g.double().t().contiguous() @ h.double()))
    assert torch.equal(ext[:, :8], g) and torch.equal(ext[:, 8:16], dh) and not ext[:, 16:].any()


def test_factors_that_do_not_fit_are_refused(K, hyc):
    """a factor of another shape, type or device raises before anything is launched, in every function that hands its address on"""
    gen = torch.Generator(device="cuda").manual_seed(4)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    M, Kf, outs, r = 20, 128, [128, 64], 16
    x, A, B, h, gs = mk(M, Kf), [mk(r, Kf) for _ in outs], [mk(o, r) for o in outs], mk(M, 2 * r), [mk(M, o) for o in outs]
    q = K.nf4_quantize(mk(sum(outs), Kf))
    for bad in ([A[0], A[1].cpu()], [A[0], mk(8, Kf)], [A[0], mk(r, 64)], [A[0], A[1].float()], [A[0], A[1].flatten()]):
        with pytest.raises(ValueError):
            K.lora_down(x, bad)
        with pytest.raises(ValueError):
            K.lora_weight_t(q, bad, outs, 64)
    for bad in ([B[0], B[1].cpu()], [B[0], mk(64, 8)], [B[0], B[1].float()], [B[1], B[0]], [B[0]], [B[0], mk(72, r)]):
        with pytest.raises(ValueError):
            K.lora_up(h, bad, 1.0, outs)
        with pytest.raises(ValueError):
            K.lora_up_bwd(gs, bad, h, 1.0, 64)
    for bad in (h[:, :r], h[:-1], h.float(), h.cpu(), mk(M, 3 * r)):
        with pytest.raises(ValueError):
            K.lora_up(bad, B, 1.0, outs) if bad.shape[0] == M else K.lora_up_bwd(gs, B, bad, 1.0, 64)
        with pytest.raises(ValueError):
            K.lora_up_bwd(gs, B, bad, 1.0, 64)
    for ext in (mk(M, 192), mk(M, 256).float(), mk(M - 1, 256), mk(M, 257)[:, :256], mk(M, 256).cpu()):
        with pytest.raises(ValueError):
            K.lora_up_bwd(gs, B, h, 1.0, 64, ext)
    for args in (([gs[0], gs[1][:-1]], B, h, 1.0, 64), ([gs[0], gs[1].cpu()], B, h, 1.0, 64), (gs, B, h, 1.0, 24)):
        with pytest.raises(ValueError):
            K.lora_up_bwd(*args)
    for args in ((q, A, outs[::-1] + [8], 64), (q, A, [128, 128], 64), (q, A, outs, 24),
                 (K.NF4Weight(q.packed[:-32], q.absmax, q.shape), A, outs, 64), (K.NF4Weight(q.packed, q.absmax.cpu(), q.shape), A, outs, 64)):
        with pytest.raises(ValueError):
            K.lora_weight_t(*args)


def test_a_group_whose_factors_do_not_fit_is_refused(K, hyc):
    """adapters on the host, of two ranks, or in the wrong order: the call raises as the products used to"""
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(2, 17, 256, generator=gen, device="cuda").bfloat16()
    for change in (lambda m: m.lora_A.cpu(), lambda m: m.lora_B.cpu(),
                   lambda m: setattr(m.lora_A[1], "data", m.lora_A[1].data[:8].clone()),
                   lambda m: [setattr(p, "data", d) for p, d in zip(m.lora_B, [m.lora_B[1].data, m.lora_B[0].data])]):
        DL, mod = _group(hyc)
        change(mod)
        with pytest.raises(ValueError):
            mod(x)
    DL, mod = _group(hyc)                                  # between forward and backward
    ys = mod(x.requires_grad_(True))
    for p, d in zip(mod.lora_B, [mod.lora_B[1].data, mod.lora_B[0].data]):
        p.data = d
    with pytest.raises((ValueError, RuntimeError)):
        torch.autograd.grad(ys, [x], [torch.ones_like(y) for y in ys])


def test_a_range_that_only_its_last_tile_takes_past_2_gib(K):
    """one range (as many feature blocks as the chip has places), whose length is rounded up to whole tiles: the general products"""
    M, out, r = 7050, 151936, 8                            # 7050 * 151936 < 2^30 <= 7104 * 151936
    gen = torch.Generator(device="cuda").manual_seed(6)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    g, h, B = mk(M, out), mk(M, r), [mk(out, r)]
    ext, dh, dB = K.lora_up_bwd([g], B, h, 0.5, 64)
    assert torch.equal(ext[:, :out], g) and torch.equal(ext[:, out:out + r], dh) and not ext[:, out + r:].any()
    close(dh[:64], 0.5 * (g[:64].float() @ B[0].float()))
    close(dB[0][:64], 0.5 * (g[:, :64].float().t().contiguous() @ h.float()))


@pytest.mark.parametrize("rank", [16, 64])                 # the kernels' and the general products' backward
def test_a_gradient_of_a_gradient(K, hyc, rank):
    """create_graph: dx and dB can be differentiated with respect to the factors and the upstream gradients, as through plain
    products (the first gradients are the ordinary ones)"""
    import importlib
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    outs = (128, 64)
    mod = DL.LoRAProjections(256, list(outs), DL.LayerConfig(hidden=256, lora_r=rank, compress=False), "cuda")
    gen = torch.Generator(device="cuda").manual_seed(7)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    x, gs, v = mk(2, 9, 256), [mk(2, 9, o) for o in outs], mk(2, 9, 256)
    plain = _gradients(mod, x, gs)
    xl, gl = x.clone().requires_grad_(True), [g.clone().requires_grad_(True) for g in gs]
    first = torch.autograd.grad(mod(xl), [xl] + list(mod.parameters()), gl, create_graph=True)
    for a, b in zip(first, plain):
        assert (a - b).abs().max() <= 4 * 2.0 ** -8 * b.abs().max()       # up to four roundings in place of one
    second = torch.autograd.grad(first[0], gl + list(mod.parameters()), v, allow_unused=True)
    A, B = ([p.detach().double().requires_grad_(True) for p in ps] for ps in (mod.lora_A, mod.lora_B))
    G = [g.double().requires_grad_(True) for g in gs]
    dx = sum(g @ (K.nf4_dequantize(w).double() + mod.scaling * b @ a) for g, w, a, b in zip(G, mod.base, A, B))
    for a, b in zip(second, torch.autograd.grad(dx, G + A + B, v.double())):
        assert (a.double() - b).norm() <= 1e-2 * b.norm()


@pytest.mark.parametrize("rank", [32, 8])
def test_factors_of_another_rank(K, hyc, rank):
    """adapters replaced by ones of another rank: the results of a group that was made with that rank"""
    import importlib
    DL = importlib.import_module(hyc.__name__ + ".decoder_layer")
    outs = (128, 64, 64)
    make = lambda r: DL.LoRAProjections(256, list(outs), DL.LayerConfig(hidden=256, lora_r=r, lora_alpha=2.0 * r, compress=False), "cuda")
    mod, want = make(16), make(rank)
    for ours, theirs in ((mod.lora_A, want.lora_A), (mod.lora_B, want.lora_B)):
        for i, p in enumerate(theirs):
            ours[i] = torch.nn.Parameter(p.detach().clone())
    mod.base_all, mod.base = want.base_all, want.base
    gen = torch.Generator(device="cuda").manual_seed(8)
    mk = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").bfloat16()
    x, gs = mk(2, 9, 256), [mk(2, 9, o) for o in outs]
    assert mod.room == K.lora_room(3, rank) == want.room
    assert all(torch.equal(a, b) for a, b in zip(_gradients(mod, x, gs), _gradients(want, x, gs)))
