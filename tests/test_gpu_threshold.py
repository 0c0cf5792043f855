"""The threshold scheme's one-chunk-per-thread kernels (csrc/threshold.hip) against the general ones: the same bytes, counts, kept elements
and results, at the edges of waves and segments, for every kind of scale and base, and where a row's slab overflows."""
import ctypes

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


def data(M, H, S, rank, kind, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + M * H + rank)
    x = torch.randn(M, H, generator=gen, device="cuda")
    x[:, ::37] *= 6
    L = torch.randn(S, rank, generator=gen, device="cuda").to(BF16) if rank else None
    R = (0.3 * torch.randn(rank, H, generator=gen, device="cuda")).to(BF16) if rank else None
    scale = {"tensor": torch.tensor(0.03), "token": 0.02 + 0.02 * torch.rand(S, 1), "channel": 0.02 + 0.02 * torch.rand(1, H)}[kind].to(BF16).cuda()
    return x.to(BF16), L, R, scale


def run_fast(hyc, K, norm, x, w, b, S, thr, scale, bits, L, R, cap):
    lib, p = hyc._abi.load(), K._p
    M, H = x.shape
    d = K.threshold_desc(thr, scale, bits, S, H, L, R)
    y, mean, rstd = torch.empty_like(x), torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    stored = torch.empty((M, H * bits // 8), dtype=torch.int8 if bits == 8 else torch.uint8, device="cuda")
    counts, slab = torch.empty(M, dtype=torch.int32, device="cuda"), torch.empty((M, cap), dtype=torch.int32, device="cuda")
    code = 0 if w is None or w.dtype == BF16 else 1
    hyc._abi.check(lib.hyc_threshold_fwd(norm, p(x), p(w), p(b), code, 1e-6, M, H, ctypes.byref(d), p(y), p(mean), p(rstd), p(stored), p(counts), p(slab),
                                         cap, K._stream()))
    row_ptr, nnz, _ = K._csr_offsets(lib, counts, M, None)
    cols, vals = torch.empty(nnz, dtype=torch.int32, device="cuda"), torch.empty(nnz, dtype=BF16, device="cuda")
    hyc._abi.check(lib.hyc_ref_outlier_fill_slab(p(x), M, H, ctypes.byref(d), p(counts), p(slab), cap, p(row_ptr), p(cols), p(vals), K._stream()))
    return y, mean, rstd, stored, row_ptr, cols, vals


@pytest.mark.parametrize("bits,M,H", [(8, 1, 64), (8, 5, 520), (8, 37, 1024), (8, 600, 1096), (8, 9, 8192), (4, 3, 128), (4, 33, 1040), (4, 2100, 768),
                                      (4, 7, 11008), (4, 5, 16384)])
@pytest.mark.parametrize("kind,rank", [("channel", 2), ("channel", 0), ("token", 1), ("tensor", 2), ("tensor", 0)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_forward_and_restore(hyc, K, bits, M, H, kind, rank, norm):
    S = 4 if M % 4 == 0 else M
    x, L, R, scale = data(M, H, S, rank, kind)
    thr, cap = 3.0, 8 if H < 1000 else 32                   # some rows keep more than the slab holds
    w = None if norm == 0 else (1 + 0.1 * torch.randn(H, device="cuda")).to(BF16 if rank else torch.float32)
    b = torch.randn_like(w) if norm == 2 and rank else None
    y, mean, rstd, *got = run_fast(hyc, K, norm, x, w, b, S, thr, scale, bits, L, R, cap)
    if norm == 0:
        c = K.compress_threshold(x, S, thr, scale, bits, L, R)
    elif norm == 1:
        y0, rstd0, c = K.rmsnorm_fwd_compress_threshold(x, w, 1e-6, S, thr, scale, bits, L, R)
        assert bits_equal(y, y0) and torch.equal(rstd, rstd0)
    else:
        y0, mean0, rstd0, c = K.layernorm_fwd_compress_threshold(x, w, b, 1e-6, S, thr, scale, bits, L, R)
        assert bits_equal(y, y0) and torch.equal(rstd, rstd0) and torch.equal(mean, mean0)
    for a, want in zip(got, (c.stored, c.row_ptr, c.cols, c.vals)):
        assert bits_equal(a, want)
    if norm == 0:
        # x_hat against the codes and entries put together in torch: bf16(bf16(base + outlier) + bf16(code * scale))
        codes = c.stored.view(torch.uint8).int()
        q = torch.cat([(codes & 15) - 8, (codes >> 4) - 8], 1) if bits == 4 else c.stored.int()
        rows = torch.repeat_interleave(torch.arange(M, device="cuda"), (c.row_ptr[1:] - c.row_ptr[:-1]).long())
        o = torch.zeros(M, H, device="cuda").index_put_((rows, c.cols.long()), c.vals.float())
        pos = torch.arange(M, device="cuda") % S
        base = torch.zeros(M, H, device="cuda")
        for r in range(rank):
            base = torch.addcmul(base.double(), L[pos, r:r + 1].double(), R[r:r + 1].double()).float()   # products of bf16 are exact, one rounding each
        base = base.to(BF16).float()
        s = scale.float()[pos] if kind == "token" else scale.float()
        want = ((base + o).to(BF16).float() + (q * s).to(BF16).float()).to(BF16)
        assert bits_equal(K.decompress_threshold(c), want)


def test_scales_outside_the_fast_range(hyc, K):
    """channels whose scale is 0, tiny or huge: the division itself, and 0 / 0 as code 0"""
    x, _, _, scale = data(16, 512, 16, 0, "channel")
    scale[0, ::5], scale[0, 1::7], scale[0, 2::11] = 0.0, 1e-35, 1e35
    x[:, ::10] = 0
    *_, stored, row_ptr, cols, vals = run_fast(hyc, K, 0, x, None, None, 16, 3.0, scale, 8, None, None, 32)
    c = K.compress_threshold(x, 16, 3.0, scale, 8)
    for a, want in zip((stored, row_ptr, cols, vals), (c.stored, c.row_ptr, c.cols, c.vals)):
        assert bits_equal(a, want)


def test_refused(hyc, K):
    for bits, H, rank in ((2, 512, 0), (8, 8256, 0), (8, 512, 3)):
        x, L, R, scale = data(8, H, 8, rank, "tensor")
        with pytest.raises(NotImplementedError):
            run_fast(hyc, K, 0, x, None, None, 8, 3.0, scale, bits, L, R, 8)
    x, L, R, scale = data(8, 512, 8, 0, "tensor")
    with pytest.raises(ValueError):
        run_fast(hyc, K, 0, x, None, None, 8, 3.0, scale, 8, L, R, 513)
