"""32-bit products by tiles chosen for the launch: every tile and the chosen one against the tile kernel through registers, bit for bit."""
import ctypes

import pytest
import torch
from test_kernels_gpu import kern, rand

pytestmark = pytest.mark.gpu
P, I, L = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
F32 = torch.float32
TILES = [(1, 1), (1, 2), (2, 2), (3, 2), (1, 4), (2, 4)]


def fine(k, x, w, M, N, K, lda, fm, fn, swiglu):
    f = k.lib.vk_gemm_fine
    f.argtypes = [P, P, P, I, I, I, L, L, I, I, I, P]
    out = torch.full((M, N), 7.0, device="cuda")
    return f(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, lda, N, fm, fn, swiglu, torch.cuda.current_stream().cuda_stream), out


@pytest.mark.parametrize("M", [1, 31, 33, 65, 97, 128, 193])
@pytest.mark.parametrize("N,K,lda", [(8, 32, 32), (66, 544, 548), (300, 1024, 1024), (1100, 96, 96), (40, 1568, 1568)])
def test_every_tile_gives_the_same_bits(M, N, K, lda):
    """Rows and columns that end inside a tile, columns that are no multiple of four, K of one pair of slabs, of whole chunks and not; more column
    blocks than a band; the product and the one with SwiGLU."""
    k = kern(F32)
    x, w = rand((M, lda), F32, 1).cuda(), rand((2 * N, K), F32, 2, 0.1).cuda()
    rows = x[:, :K].contiguous()
    want, up = k.gemm(rows, w[:N].contiguous(), kernel=3), k.gemm(rows, w[N:].contiguous(), kernel=3)
    gated = (want.double() * torch.sigmoid(want.double()) * up.double())
    first = None
    for fm, fn in TILES + [(0, 0)]:
        rc, out = fine(k, x, w, M, N, K, lda, fm, fn, 0)
        assert rc == 0 and torch.equal(out, want), (fm, fn)
        if fn == 1:
            continue
        rc, out = fine(k, x, w, M, N, K, lda, fm, fn, 1)
        # an exponential, a sum, a quotient and two products, each within two units in the last place (1.2e-7)
        assert rc == 0 and torch.allclose(out.double(), gated, rtol=1.2e-6, atol=1e-30), (fm, fn)
        first = out if first is None else first
        assert torch.equal(out, first), (fm, fn)


# Few rows of K that is no whole number of chunks: the streaming kernels where weight rows are few, small tiles where tiles of 128 rows
# would fill half of the units; many rows: larger tiles where they fill the units' rounds.
@pytest.mark.parametrize("M,N,K,small", [(33, 1024, 1280, 0), (48, 4096, 1504, 0), (49, 1024, 1280, 1), (33, 4112, 1280, 1), (64, 16256, 1568, 0), (33, 16288, 1568, 1), (64, 16384, 2080, 1),
                                         (33, 1024, 1536, 1), (64, 1024, 2048, 0), (512, 10240, 2080, 0), (1024, 8192, 544, 0), (2048, 4096, 544, 0), (256, 20480, 1024, 0),
                                         (200, 4096, 2080, 1), (651, 2048, 6144, 1), (128, 8192, 1024, 1)])
def test_which_tiles_and_their_bits(M, N, K, small):
    k = kern(F32)
    x, w = rand((M, K), F32, 1).cuda(), rand((N, K), F32, 2, 0.1).cuda()
    takes = k.lib.vk_gemm_fine_takes
    takes.argtypes = [I, I, I, L, I]
    assert takes(M, N, K, K, 0) == small
    assert torch.equal(k.gemm(x, w), k.gemm(x, w, kernel=3))


@pytest.mark.parametrize("M,I_,K,small", [(512, 8192, 544, 0), (1024, 4096, 1024, 0), (434, 4096, 544, 1), (65, 4096, 544, 1)])
def test_which_tiles_with_swiglu(M, I_, K, small):
    k = kern(F32)
    takes = k.lib.vk_gemm_fine_takes
    takes.argtypes = [I, I, I, L, I]
    assert takes(M, I_, K, K, 1) == small
    x, w = rand((M, K), F32, 1).cuda(), rand((2 * I_, K), F32, 2, 0.1).cuda()
    f = k.lib.vk_gemm_swiglu
    f.argtypes = [P, P, P, I, I, I, L, L, P]
    out = torch.empty(M, I_, device="cuda")
    assert f(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, I_, K, K, I_, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, k.swiglu(k.gemm(x, w, kernel=3)))


@pytest.mark.parametrize("M,I_,K", [(33, 200, 512), (64, 96, 1024), (65, 200, 96), (300, 1000, 512)])
def test_swiglu_by_size_is_the_product_and_the_activation(M, I_, K):
    k = kern(F32)
    x, w = rand((M, K), F32, 1).cuda(), rand((2 * I_, K), F32, 2, 0.1).cuda()
    f = k.lib.vk_gemm_swiglu
    f.argtypes = [P, P, P, I, I, I, L, L, P]
    out = torch.empty(M, I_, device="cuda")
    assert f(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, I_, K, K, I_, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, k.swiglu(k.gemm(x, w, kernel=3)))


def test_what_is_refused():
    k = kern(F32)
    x, w = torch.zeros(64, 64, device="cuda"), torch.zeros(128, 64, device="cuda")
    assert fine(k, x, w, 64, 64, 64, 64, 5, 5, 0)[0] != 0          # no such tile
    assert fine(k, x, w, 64, 64, 64, 64, 1, 1, 1)[0] != 0          # no gate and up fragments in one
    assert fine(k, x, w, 64, 64, 48, 64, 1, 1, 0)[0] != 0          # K not in whole pairs of slabs
    half = kern(torch.bfloat16)
    assert fine(half, x, w, 64, 64, 64, 64, 1, 1, 0)[0] != 0
