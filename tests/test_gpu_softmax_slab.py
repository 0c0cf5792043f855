"""Kept probabilities through the forward's slab against the form that reads the probabilities a second time: the same
probabilities, offsets, columns and values, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import importlib
    return importlib.import_module("hyc-lora_amd").kernels


# chunks per lane 1, 2, 4, 8 with whole and cut rows; rows around the 4096 of an offsets workgroup
@pytest.mark.parametrize("rows,N", [(1, 64), (7, 256), (64, 504), (33, 512), (4096, 520), (4097, 1024), (8200, 1000), (130, 2048), (70, 2040),
                                    (65, 4096), (66, 3000)])
@pytest.mark.parametrize("causal,keep,seen", [(False, 0.01, 1.0), (True, 0.01, 1.0), (False, 0.2, 0.05), (True, 1.0, 0.01)])
def test_slab_matches_second_read(K, rows, N, causal, keep, seen):
    """seen: the share of the true one that the budget has seen (small: most rows overflow the slab and are read again)"""
    gen = torch.Generator().manual_seed(rows + N)
    x = (2 * torch.randn(rows, N, generator=gen)).bfloat16().cuda()
    period = N if causal else None
    y0, _ = K.softmax_fwd(x, causal_period=period)
    thr = -1.0 if keep == 1.0 else float(torch.quantile(y0[:64].float().flatten()[:1 << 20].cpu(), 1 - keep))
    y1, want = K.softmax_fwd(x, thr, causal_period=period)
    assert torch.equal(y0, y1)
    budget = K.KeptBudget()
    budget.observe(max(1.0, seen * want.cols.numel()), rows)
    cap = K._slab_entries(budget, N)
    budget.capacity = lambda n: want.cols.numel() + 64                # room for all, whatever the share seen
    for inplace in (False, True):
        xi = x.clone()
        y, got = K.softmax_fwd(xi, thr, causal_period=period, inplace=inplace, budget=budget)
        budget._pending.clear()
        assert cap > 0 or N < 256 or keep > 0.1
        assert torch.equal(y, y0)
        n = want.cols.numel()
        assert int(got.total) == n and torch.equal(got.row_ptr, want.row_ptr)
        assert torch.equal(got.cols[:n], want.cols) and torch.equal(got.vals[:n].view(torch.int16), want.vals.view(torch.int16))


def test_slab_keeps_to_the_capacity(K):
    """offsets cut off at the capacity: no entry lands behind it, and the total tells"""
    rows, N = 300, 1024
    x = torch.randn(rows, N, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    _, want = K.softmax_fwd(x, 4.0 / N)
    room = want.cols.numel() // 2
    budget = K.KeptBudget()
    budget.observe(32 * rows, rows)
    budget.capacity = lambda n: room
    _, got = K.softmax_fwd(x, 4.0 / N, budget=budget)
    budget._pending.clear()
    assert got.cols.numel() == room and int(got.total) == want.cols.numel()
    assert torch.equal(got.cols, want.cols[:room]) and int(got.row_ptr[-1]) == room
