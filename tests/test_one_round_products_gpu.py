"""Tile products whose workgroups are at most as many as the compute units: the bits of the two-stage square tiles on both sides of each line."""
import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K", [64, 128, 192, 512, 576, 1024, 1536, 2112])
@pytest.mark.parametrize("M", [65, 128, 129, 257, 641])
def test_widths_of_one_round(M, K, dtype):
    """The widest product that fits with 64, 96 and 128 weight rows a workgroup, one more weight row than that, and one that ends inside the first
    workgroup; fewer tiles of K than stages, and K in whole chunks and not.  Rows further apart than they are long."""
    k = kern(dtype)
    cus, blocks = torch.cuda.get_device_properties(0).multi_processor_count, -(-M // 128)
    x = rand((M, K + 32), dtype, 1).cuda()[:, :K]
    for N in [7, 200] + [width * (cus // blocks) + more for width in (64, 96, 128) for more in (0, 1)]:
        w = rand((N, K), dtype, 2, 0.1).cuda()
        assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=4)), N


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K", [64, 128, 576, 1024])
@pytest.mark.parametrize("M", [65, 128, 300, 641])
def test_gate_and_up(M, K, dtype):
    k = kern(dtype)
    cus, blocks = torch.cuda.get_device_properties(0).multi_processor_count, -(-M // 128)
    x = rand((M, K), dtype, 3).cuda()
    for I in (7, 200, 64 * (cus // blocks), 64 * (cus // blocks) + 1):
        w = rand((2 * I, K), dtype, 4, 0.1).cuda()
        assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4))), I


@pytest.mark.parametrize("M", [112, 113, 128, 129])
@pytest.mark.parametrize("K", [4608, 5120])
def test_a_second_block_of_rows(M, K):
    """Both sides of the lines in rows, chunks and weight rows at which 16-bit products of two blocks of 64 rows share activations through LDS instead."""
    k = kern(torch.bfloat16)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    x = rand((M, K), torch.bfloat16, 7).cuda()
    for N in (16 * cus, 16 * cus + 1, 32 * cus, 32 * cus + 1):
        w = (torch.randn((N, K), generator=torch.Generator("cuda").manual_seed(8), device="cuda") * 0.1).to(torch.bfloat16)
        assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=4)), N


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_far_apart(dtype):
    """Rows whose distance from the first of their block is no longer a number of 32 bits in bytes: 127 of them are more than 4 GiB, by 23 MB."""
    k = kern(dtype)
    M, K, apart = 128, 512, 17_000_000 if dtype == torch.bfloat16 else 8_500_000
    rows = rand((M, K), dtype, 5).cuda()
    x = torch.empty(((M - 1) * apart + K,), dtype=dtype, device="cuda").as_strided((M, K), (apart, 1))
    x.copy_(rows)
    w = rand((512, K), dtype, 6, 0.1).cuda()
    expected = k.gemm(rows, w, kernel=3)
    assert torch.equal(k.gemm(x, w), expected) and torch.equal(k.gemm(x, w, kernel=2), expected)
    assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(expected))
