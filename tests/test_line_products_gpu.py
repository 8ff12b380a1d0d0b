"""Products of up to 16 rows whose weights come through LDS in whole lines: the bits of the tile kernel, by name and as chosen by size."""
import pytest
import torch
from test_kernels_gpu import kern, rand

pytestmark = pytest.mark.gpu
B = torch.bfloat16


def weights(shape, seed):
    return (torch.randn(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda") * 0.1).to(B)


@pytest.mark.parametrize("chunks", [1, 2, 3, 5, 8, 9, 12])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16])
def test_tiles_and_rings(M, chunks):
    """Weight rows that end inside a tile and are no multiple of four, fewer tiles than a ring has slots, and many more; rows further apart than they are long."""
    k = kern(B)
    K = 512 * chunks
    x = rand((M, K + 32), B, 1).cuda()[:, :K]
    for N in (1, 7, 300, 2049, 9001):
        w = weights((N, K), 2)
        expected = k.gemm(x, w, kernel=4)
        assert torch.equal(k.gemm(x, w), expected), N
        if M <= 8 or chunks <= 8:
            assert torch.equal(k.gemm(x, w, kernel=20), expected) and torch.equal(k.gemm(x, w, kernel=21), expected), N


@pytest.mark.parametrize("chunks", [2, 4, 5, 7, 8, 10, 12])
@pytest.mark.parametrize("M", [1, 3, 8, 9, 16])
def test_gate_and_up(M, chunks):
    """On both sides of the lines at half a compute unit's worth of tiles and a whole one."""
    k = kern(B)
    K = 512 * chunks
    x = rand((M, K), B, 3).cuda()
    for I in (24, 2040, 2056, 4104, 13000):
        w = weights((2 * I, K), 4)
        assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4))), I


def test_sizes_that_do_not_fit():
    from vosti_amd.kernels.ops import KernelError
    k = kern(B)
    w = weights((64, 512 * 13), 5)
    for rows, chunks in ((17, 2), (16, 12), (1, 13)):
        with pytest.raises(KernelError):
            k.gemm(rand((rows, 512 * chunks), B, 6).cuda(), w[:, :512 * chunks].contiguous(), kernel=21)
    with pytest.raises(KernelError):
        kern(torch.float32).gemm(torch.zeros(1, 512, device="cuda"), torch.zeros(8, 512, device="cuda"), kernel=20)


@pytest.mark.parametrize("N,K", [(1449, 800), (1702, 1024), (1393, 1184), (1301, 1536), (1500, 2048), (1100, 2336), (700, 3072), (699, 3104), (700, 4096), (64, 8192)])
def test_experts(N, K):
    """Experts' products from the line on at which their weights come in whole lines, for every number of chunks, whole and not; features that end inside a
    group of eight."""
    from test_expert_tiles_gpu import test_tiles_get_the_plain_product
    test_tiles_get_the_plain_product(N, K, B)
