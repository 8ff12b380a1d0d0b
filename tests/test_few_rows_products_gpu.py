"""Products of 17 to 64 rows whose weights come through LDS in lines: the bits of the tile kernel on both sides of every line of the rule."""
import pytest
import torch
from test_kernels_gpu import kern, rand

pytestmark = pytest.mark.gpu
B = torch.bfloat16


def weights(shape, seed):
    return (torch.randn(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda") * 0.1).to(B)


@pytest.mark.parametrize("chunks", [1, 2, 4, 5, 8, 9])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 64])
def test_plain(M, chunks):
    """Weight rows that end inside a wave's sixteen and are no multiple of four; rows further apart than they are long; with and without a workspace."""
    k = kern(B)
    K, cus = 512 * chunks, torch.cuda.get_device_properties(0).multi_processor_count
    x = rand((M, K + 32), B, 1).cuda()[:, :K]
    for N in (16 * cus, 16 * cus + 1, 24 * cus - 35, 24 * cus, 28 * cus + 33, 32 * cus, 32 * cus + 1, 64 * cus + 70):
        w = weights((N, K), 2)
        expected = k.gemm(x, w, kernel=4)
        assert torch.equal(k.gemm(x, w), expected), N
        need = k.gemm_workspace_floats(M, N, K)
        if need:
            assert torch.equal(k.gemm(x, w, workspace=torch.empty(need, device="cuda")), expected), N


@pytest.mark.parametrize("chunks", [1, 4, 5, 8, 10])
@pytest.mark.parametrize("M", [17, 32, 33, 64])
def test_gate_and_up(M, chunks):
    k = kern(B)
    K, cus = 512 * chunks, torch.cuda.get_device_properties(0).multi_processor_count
    x = rand((M, K), B, 3).cuda()
    for I in (7, 300, 16 * cus, 16 * cus + 1, 28 * cus + 33, 32 * cus, 32 * cus + 3, 64 * cus, 64 * cus + 1, 96 * cus + 40):
        w = weights((2 * I, K), 4)
        assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4))), I
