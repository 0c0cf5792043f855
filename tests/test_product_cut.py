"""Where the decoder layer cuts a product with the library's kernels in two (no GPU needed)."""
import importlib

import pytest
import torch

DL = importlib.import_module("hyc-lora_amd.decoder_layer")


def rounds(M, N):
    return -(-(-(-M // 256) * -(-N // 256)) // 256)


def test_a_cut_adds_no_round():
    for N in list(range(256, 40000, 256)) + [8200, 11000, 5003]:
        for M in (1, 157, 1024, 1300, 1536, 2048, 2304, 2560, 3093, 4096, 5120, 8192, 16384):
            cut = DL._cut_columns(M, N)
            assert cut in (0, 4096, 8192) and cut < N
            if cut:
                assert N % 256 == 0 and N % 4096 and rounds(M, cut) + rounds(M, N - cut) <= rounds(M, N)


@pytest.mark.parametrize("M,N,cut", [(2048, 22016, 8192), (4096, 22016, 8192), (2560, 22016, 0), (5120, 22016, 0), (2048, 11008, 8192), (2560, 11008, 0),
                                     (4096, 5632, 4096), (2048, 5632, 0), (2048, 8448, 8192), (2560, 8448, 0), (2048, 13824, 0), (2048, 27648, 0),
                                     (4096, 14336, 0), (4096, 4096, 0), (4096, 12288, 0), (4096, 2048, 0), (0, 22016, 0)])
def test_cut_of_measured_widths(M, N, cut):
    assert DL._cut_columns(M, N) == cut


@pytest.mark.parametrize("accumulate", [False, True])
def test_a_cut_product_is_the_product(accumulate):
    M, N, K = 4096, 4608, 8
    assert DL._cut_columns(M, N) == 4096
    gen = torch.Generator().manual_seed(0)
    a, b = (torch.randint(-3, 4, s, generator=gen).bfloat16() for s in ((M, K), (N, K)))
    start = torch.randint(-3, 4, (M, N), generator=gen).bfloat16()
    out = start.clone()
    DL._product(out, a, b, accumulate)
    want = a.float() @ b.float().t() + (start.float() if accumulate else 0)     # small whole numbers: exact in bf16
    assert torch.equal(out.float(), want)
