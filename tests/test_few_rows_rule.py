"""Where dX over few tokens is taken by the package's own kernel: while a launch's workgroups, one a CU, are resident at once (no GPU needed)."""
import importlib

import pytest

A = importlib.import_module("hyc-lora_amd")._abi


@pytest.fixture(scope="module")
def covers():
    if not A.built():
        pytest.skip("the kernel library is not built")
    return lambda M, K, N: A.load().hyc_few_rows_covers(M, K, N, 1)


@pytest.mark.parametrize("N,K,last", [(11008, 4160, 80), (5632, 2112, 160), (2816, 1088, 320), (1536, 4160, 640)])
def test_a_second_round_is_the_librarys(covers, N, K, last):
    assert covers(last, K, N) and not covers(last + 1, K, N) and not covers((1 << 20) // N, K, N)


def test_a_single_block_of_tokens_and_the_bounds(covers):
    for M, K, N in ((16, 4160, 22016), (47, 4160, 22016), (32, 4160, 32768), (16, 512, 65536), (75, 5184, 13824), (157, 11328, 2048), (512, 1088, 2048),
                    (256, 12352, 4096), (1024, 11072, 1024)):
        assert covers(M, K, N)
    for M, K, N in ((76, 4160, 13824), (48, 4160, 22016), (513, 1088, 2048), (1025, 64, 16), (257, 4096, 4096)):
        assert not covers(M, K, N)
