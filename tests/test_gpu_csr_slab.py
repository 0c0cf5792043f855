"""Row offsets and the copy of a slab of kept entries in one launch against the two: rows around a workgroup's four, a step of the counts'
sum (1024) and the limit of the one launch; entries cut off at a capacity; rows of more entries than the slab holds, which are read again."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


def pointers(ts):
    return [t.data_ptr() for t in ts]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("share", [0.3, 1.0])
@pytest.mark.parametrize("rows", [1, 3, 4, 5, 1023, 1024, 1029, 4097, 8192, 8193])
def test_one_launch(K, rows, share, offset):
    lib, N, cap, limit = K._abi.load(), 64, 6, 1.25
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, N, generator=gen, device="cuda").to(BF16)
    x[0] = 3.0                                              # (a row of which everything is kept)
    hot = x > limit                                         # (of the outliers |x| > limit; see below)
    for kind in ("softmax", "outlier"):
        mask = hot if kind == "softmax" else x.abs() > limit
        counts = torch.zeros(rows + 1, dtype=torch.int32, device="cuda")[offset:][:rows]   # (an odd address takes the two launches)
        counts.copy_(mask.sum(1))
        order = torch.sort((~mask).to(torch.int8), dim=1, stable=True).indices[:, :cap]     # the kept columns first, in their order
        bits = torch.gather(x, 1, order).view(torch.int16).to(torch.int32) & 0xFFFF
        slab = (order.to(torch.int32) | bits << 16).contiguous()
        total = int(counts.sum())
        capacity = max(1, int(share * total))
        new = lambda: (torch.full((rows + 1,), -1, dtype=torch.int32, device="cuda"), torch.zeros((), dtype=torch.int64, device="cuda"),
                       torch.full((capacity + 1,), -1, dtype=torch.int32, device="cuda"), torch.full((capacity + 1,), -1, dtype=torch.int16, device="cuda"))
        a, b = new(), new()
        (ra, ta, ca, va), (rb, tb, cb, vb) = pointers(a), pointers(b)
        K.check(lib.hyc_csr_offsets(counts.data_ptr(), rows, capacity, ra, ta, K._stream()))
        if kind == "softmax":
            K.check(lib.hyc_softmax_fill_slab(x.data_ptr(), rows, N, limit, counts.data_ptr(), slab.data_ptr(), cap, ra, ca, va, K._stream()))
            K.check(lib.hyc_softmax_csr_slab(x.data_ptr(), rows, N, limit, counts.data_ptr(), slab.data_ptr(), cap, capacity, rb, tb, cb, vb, K._stream()))
        else:
            scale = torch.ones(1, dtype=BF16, device="cuda")
            d = K.threshold_desc(limit, scale, 8, rows, N, None, None, None, None, None)
            K.check(lib.hyc_ref_outlier_fill_slab(x.data_ptr(), rows, N, ctypes.byref(d), counts.data_ptr(), slab.data_ptr(), cap, ra, ca, va, K._stream()))
            K.check(lib.hyc_ref_outlier_csr_slab(x.data_ptr(), rows, N, ctypes.byref(d), counts.data_ptr(), slab.data_ptr(), cap, capacity, rb, tb, cb, vb,
                                                 K._stream()))
        torch.cuda.synchronize()
        assert all(torch.equal(s, t) for s, t in zip(a, b))
        ends = torch.cat([counts.new_zeros(1), counts.cumsum(0)]).clamp(max=capacity)
        assert torch.equal(b[0], ends.to(torch.int32)) and int(b[1]) == total and int(b[2][-1]) == -1
        assert torch.equal(b[2][:-1], mask.nonzero()[:capacity, 1].to(torch.int32)) and torch.equal(b[3][:-1].view(BF16), x[mask][:capacity])
