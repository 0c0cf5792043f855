"""What the LoRA functions check about a group's factors before an address leaves Python (no GPU needed)."""
import importlib

import pytest
import torch

K = importlib.import_module("hyc-lora_amd").kernels
CPU = torch.device("cpu")


def factors(*shapes, dtype=torch.bfloat16):
    return [torch.zeros(s, dtype=dtype) for s in shapes]


def test_factors_must_have_their_shape_type_and_device():
    shapes = [(16, 128), (16, 128)]
    assert K._lora_factors(factors(*shapes), shapes, CPU, "A") is True
    for bad in (factors((16, 128), (8, 128)), factors((16, 128), (16, 64)), factors((16, 128)), factors((16, 128), (2048,)),
                factors(*shapes, dtype=torch.float32), [torch.zeros(16, 128, dtype=torch.bfloat16), None],
                [torch.zeros(16, 128, dtype=torch.bfloat16), torch.zeros(16, 128, dtype=torch.bfloat16, device="meta")]):
        with pytest.raises(ValueError):
            K._lora_factors(bad, shapes, CPU, "A")
    with pytest.raises(ValueError):                        # the second factor of a swapped pair
        K._lora_factors(factors((64, 16), (128, 16)), [(128, 16), (64, 16)], CPU, "B")


def test_factors_the_kernels_cannot_read_as_they_lie_go_elsewhere():
    assert K._lora_factors([torch.zeros(128, 16, dtype=torch.bfloat16).t()], [(16, 128)], CPU, "A") is False
    assert K._lora_factors([torch.zeros(16 * 128 + 1, dtype=torch.bfloat16)[1:].view(16, 128)], [(16, 128)], CPU, "A") is False


def test_token_ranges_are_bounded_with_their_last_tile():
    fits = K._lora_range_fits
    for M, pitch in ((7041, 151936), (7050, 151936), (7067, 151936)):          # the last tile takes the range past 2^30 elements
        assert M * pitch < 1 << 30 <= (M + 63) // 64 * 64 * pitch and not fits(M, pitch)
    assert fits(7040, 151936) and fits(1 << 20, 32760) and not fits(1 << 20, 32768) and fits(1, 1 << 23) and not fits(1, 1 << 24)


def test_sizes_past_what_a_launch_counts_take_the_general_products():
    cover = K._lora_kernels_cover
    assert cover(4096, 3, 16, 4096, (4096,) * 3) and cover(65535 * 128, 1, 8, 64, (8,))
    for args in ((65535 * 128 + 1, 1, 8, 64, (8,)), (1, 1, 8, 64, (65535 * 128,)), (1, 1, 8, (1 << 24) + 64, (8,)), (1, 5, 8, 64, (8,) * 5),
                 (1, 1, 64, 64, (8,)), (1, 1, 8, 32, (8,)), (1, 1, 8, 64, (12,)), (1, 2, 8, 64, (8, 0))):
        assert not cover(*args)
