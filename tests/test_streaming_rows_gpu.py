"""Products of up to 16 rows whose activations come through LDS: the bits of the tile kernel."""
import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunks", [1, 2, 3, 5, 6, 8, 9, 10, 12, 13, 19])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16])
def test_rows_and_chunks(M, chunks, dtype):
    """One row to 16, waves with a chunk, with several and without one, weight rows that end inside a tile; rows further apart than they are
    long."""
    k = kern(dtype)
    K = 512 * chunks
    x = rand((M, K + 32), dtype, 1).cuda()[:, :K]
    for N in (9, 300, 4200 if chunks > 3 else 17000):
        w = rand((N, K), dtype, 2, 0.1).cuda()
        assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=4)), N


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunks", [1, 2, 4, 5, 6, 8])
@pytest.mark.parametrize("M", [1, 3, 8, 9, 16])
def test_gate_and_up(M, chunks, dtype):
    k = kern(dtype)
    K = 512 * chunks
    x = rand((M, K), dtype, 3).cuda()
    for I in (24, 4200):
        w = rand((2 * I, K), dtype, 4, 0.1).cuda()
        assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4)))


@pytest.mark.parametrize("M,I,K", [(17, 12300, 512), (24, 8201, 1024), (32, 4097, 4096), (20, 16, 2048), (31, 4096, 2560)])
def test_gate_and_up_of_two_tiles_of_rows(M, I, K):
    """17 to 32 rows: several weight tiles a workgroup and one, the last of them partial, waves without a chunk."""
    k = kern(torch.bfloat16)
    x, w = rand((M, K), torch.bfloat16, 5).cuda(), rand((2 * I, K), torch.bfloat16, 6, 0.1).cuda()
    assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N", [3072, 3088, 4090, 4096, 4097])
@pytest.mark.parametrize("M", [8, 9, 16])
def test_two_chunks_and_about_a_weight_tile_a_compute_unit(M, N, dtype):
    """On both sides of the line between rows through LDS and rows straight to registers."""
    k = kern(dtype)
    x, w = rand((M, 1024), dtype, 7).cuda(), rand((N, 1024), dtype, 8, 0.1).cuda()
    assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=4))


def rows_of_several_tiles(waves):
    """Weight rows that give a workgroup of `waves` waves more than one tile, however many of them run at once (a compute unit holds 32 waves)."""
    return 16 * torch.cuda.get_device_properties(0).multi_processor_count * (32 // waves) + 9


def weights(shape, dtype, seed):
    return (torch.randn(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda") * 0.1).to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunks,waves", [(1, 2), (2, 2), (4, 4), (5, 5), (6, 6), (8, 8), (10, 8), (12, 8), (19, 8)])
@pytest.mark.parametrize("M", [1, 4, 8, 16])
def test_more_tiles_than_workgroups(M, chunks, waves, dtype):
    """A workgroup's first tile, one in between and its last: what it streams from one to the next, and the rows a chunk ahead that are those of the next
    tile's first chunk."""
    k = kern(dtype)
    x, w = rand((M, 512 * chunks), dtype, 9).cuda(), weights((rows_of_several_tiles(waves), 512 * chunks), dtype, 10)
    assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=4))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunks,waves", [(1, 2), (2, 2), (4, 4), (5, 5), (6, 6), (8, 8), (10, 8), (12, 8)])
@pytest.mark.parametrize("M", [1, 4, 8, 16])
def test_gate_and_up_with_more_tiles_than_workgroups(M, chunks, waves, dtype):
    k = kern(dtype)
    x, w = rand((M, 512 * chunks), dtype, 11).cuda(), weights((2 * rows_of_several_tiles(waves), 512 * chunks), dtype, 12)
    assert torch.equal(k.gemm_swiglu(x, w), k.swiglu(k.gemm(x, w, kernel=4)))
