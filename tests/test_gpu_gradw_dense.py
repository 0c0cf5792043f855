"""The weight gradient of a dense activation on 256 x 256 tiles, where its pipeline can go wrong: token ranges of fewer stages than
it has buffers, that are cut within a stage or fill whole rounds of buffers, split ranges, feature tiles cut at every eighth
column, outputs in both types and on top of what is there, and operands whose neighbours in memory are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(hyc):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return hyc.kernels


@pytest.mark.parametrize("M", [1, 31, 32, 33, 95, 96, 97, 128, 130, 161, 511, 777, 2080])
@pytest.mark.parametrize("N,H", [(256, 256), (264, 512), (520, 256), (1024, 1024)])
def test_dense_weight_gradient(K, M, N, H):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    # whole numbers whose sums stay below 2^24: exact in fp32 in any order
    wide = torch.full((M + 2, N + 16), float("nan"), device="cuda").bfloat16()
    wide[1:M + 1, 8:N + 8] = torch.randint(-8, 9, (M, N), generator=gen, device="cuda").bfloat16()
    dy = wide[1:M + 1, 8:N + 8]
    tall = torch.full((M + 2, H), float("nan"), device="cuda").bfloat16()
    tall[1:M + 1] = torch.randint(-8, 9, (M, H), generator=gen, device="cuda").bfloat16()
    x = tall[1:M + 1]
    want = dy.float().t().contiguous() @ x.float()
    got = K.gradw_gemm(dy, x, out_dtype=torch.float32)
    assert torch.equal(got, want)
    assert torch.equal(K.gradw_gemm(dy, x, out_dtype=torch.bfloat16), want.bfloat16())
    base = torch.ones(N, H, device="cuda")
    assert torch.equal(K.gradw_gemm(dy, x, alpha=2.0, out=base, beta=0.5), 2 * want + 0.5)
