"""The tile product whose two groups of waves take turns: the bits of the tile kernel, at the edges of its tiles."""
import ctypes

import pytest
import torch
from test_kernels_gpu import kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [192, 160, 128])
@pytest.mark.parametrize("M,extra,K,lda", [(256, 0, 512, 512), (257, 1, 1024, 1032), (511, -1, 512, 520), (700, 67, 1536, 1536), (1030, 1500, 512, 512)])
def test_same_bits_as_the_tile_kernel(M, extra, K, lda, columns):
    """One whole tile, a row and a column more, one fewer than two, blocks that overlap the one before by almost all of it, and bands of
    more and fewer than eight column blocks; one chunk of K and several; rows further apart than they are long."""
    k = kern(torch.bfloat16)
    N = columns + extra if extra >= 0 else 2 * columns + extra
    act, w = rand((M, lda), torch.bfloat16, 1).cuda()[:, :K], rand((N, K), torch.bfloat16, 2, 0.1).cuda()
    want = k.gemm(act, w, kernel=4)
    code = {192: 17, 160: 18, 128: 19}[columns]
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert torch.equal(k.gemm(act, w, out=out, kernel=code), want)
    # Rows of the output further apart than they are long and on odd addresses: element by element, nothing beyond a row's end.
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_gemm
    fn.argtypes = [p, p, p, i, i, i, l, l, i, p]
    wide = torch.full((M * (N + 3) + 1,), 7.0, dtype=torch.bfloat16, device="cuda")
    assert fn(wide.data_ptr() + 2, act.data_ptr(), w.data_ptr(), M, N, K, lda, N + 3, code, torch.cuda.current_stream().cuda_stream) == 0
    rows = wide[1:].view(M, N + 3)
    assert torch.equal(rows[:, :N], want) and bool((rows[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,I,K", [(256, 4096, 512), (2048, 3072, 1024), (513, 1633, 1024), (300, 12288, 512)])
def test_gate_and_up_by_size(M, I, K):
    """The product with SwiGLU folded in, its kernel chosen by size, against the plain product and the activation."""
    k = kern(torch.bfloat16)
    act, w = rand((M, K), torch.bfloat16, 3).cuda(), rand((2 * I, K), torch.bfloat16, 4, 0.1).cuda()
    assert torch.equal(k.gemm_swiglu(act, w), k.swiglu(k.gemm(act, w, kernel=4)))


@pytest.mark.parametrize("M,N,K", [(2048, 6144, 512), (1500, 5120, 1024), (3333, 4096, 512), (1024, 4100, 2048), (255, 8192, 512)])
def test_product_by_size(M, N, K):
    """Sizes on both sides of the rule that chooses between the kernels."""
    k = kern(torch.bfloat16)
    act, w = rand((M, K), torch.bfloat16, 5).cuda(), rand((N, K), torch.bfloat16, 6, 0.1).cuda()
    assert torch.equal(k.gemm(act, w), k.gemm(act, w, kernel=4))


@pytest.mark.parametrize("M,N,K", [(256, 195, 512), (700, 1633, 1024), (2048, 4097, 512), (511, 4099, 1024), (300, 4102, 512)])
def test_columns_that_are_no_multiple_of_four(M, N, K):
    """Rows of the output on whole vectors, a last block of columns that does not begin on one: every store on its type's alignment, nothing beyond a row's
    end, plain and with SwiGLU folded in."""
    k = kern(torch.bfloat16)
    ldo = (N + 7) // 4 * 4
    act, w = rand((M, K), torch.bfloat16, 9).cuda(), rand((2 * N, K), torch.bfloat16, 10, 0.1).cuda()
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    k.lib.vk_gemm.argtypes = [p, p, p, i, i, i, l, l, i, p]
    k.lib.vk_gemm_swiglu.argtypes = [p, p, p, i, i, i, l, l, p]
    stream = torch.cuda.current_stream().cuda_stream
    plain, gated = k.gemm(act, w[:N], kernel=4), k.swiglu(k.gemm(act, w, kernel=4))
    for code in (0, 17, 18, 19):
        out = torch.full((M, ldo), 7.0, dtype=torch.bfloat16, device="cuda")
        assert k.lib.vk_gemm(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, K, ldo, code, stream) == 0
        assert torch.equal(out[:, :N], plain) and bool((out[:, N:] == 7.0).all()), code
    out = torch.full((M, ldo), 7.0, dtype=torch.bfloat16, device="cuda")
    assert k.lib.vk_gemm_swiglu(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, K, ldo, stream) == 0
    assert torch.equal(out[:, :N], gated) and bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(2048, 6144, 512), (3333, 4096, 512), (2048, 6150, 512), (1500, 5123, 1024)])
def test_squared_relu_by_size(M, N, K):
    """The activation in the epilogue, blocks that overlap the one before among them (they are computed and stored twice)."""
    k = kern(torch.bfloat16)
    act, w = rand((M, K), torch.bfloat16, 12).cuda(), rand((N, K), torch.bfloat16, 13, 0.1).cuda()
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    k.lib.vk_gemm_act.argtypes = [p, p, p, i, i, i, l, l, i, p]
    for ldo in (N, (N + 7) // 4 * 4):
        out = torch.full((M, ldo), 7.0, dtype=torch.bfloat16, device="cuda")
        assert k.lib.vk_gemm_act(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, K, ldo, 1, torch.cuda.current_stream().cuda_stream) == 0
        r = k.gemm(act, w, kernel=4).float().clamp(min=0)
        assert torch.equal(out[:, :N], (r * r).to(torch.bfloat16)) and bool((out[:, N:] == 7.0).all())


def test_sizes_below_a_tile_are_refused():
    k = kern(torch.bfloat16)
    w = rand((256, 512), torch.bfloat16, 7).cuda()
    for code, rows, M, K in ((17, 191, 256, 512), (18, 159, 256, 512), (19, 128, 255, 512), (19, 128, 256, 448)):
        with pytest.raises(Exception, match="alternating"):
            k.gemm(rand((M, K), torch.bfloat16, 8).cuda(), w.flatten()[: rows * K].view(rows, K), kernel=code)


@pytest.mark.parametrize("code", [17, 18, 19])
@pytest.mark.parametrize("M", [0, 256])
def test_32_bit_elements_are_refused(M, code):
    k = kern(torch.float32)
    x = rand((256, 512), torch.float32, 11).cuda()
    with pytest.raises(Exception, match="unknown kernel"):
        k.gemm(x[:M], x, kernel=code)
