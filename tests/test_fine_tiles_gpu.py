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
@pytest.mark.parametrize("N,K,lda", [(8, 32, 32), (66, 544, 548), (300, 1024, 1024), (1100, 96, 96)])
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
