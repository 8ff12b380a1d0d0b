"""Products that add and norm their rows themselves: the bits of the norm and the product by themselves."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu
P, I = ctypes.c_void_p, ctypes.c_int


def normed(k, x, residual, weight, eps, w, projections):
    M, K = x.shape
    N = w.shape[0] // projections
    takes, run = k.lib.vk_gemm_normed_takes, k.lib.vk_gemm_normed
    takes.argtypes = [I, I, I, I]
    run.argtypes = [P, P, P, P, P, ctypes.c_float, P, I, I, I, ctypes.c_int64, I, P]
    out, total = torch.full((M, N), float("nan"), dtype=x.dtype, device="cuda"), torch.full_like(x, float("nan"))
    rc = run(out.data_ptr(), total.data_ptr(), x.data_ptr(), residual.data_ptr(), weight.data_ptr(), eps, w.data_ptr(), M, N, K, N, projections,
             torch.cuda.current_stream().cuda_stream)
    assert (rc == 0) == bool(takes(M, N, K, projections))
    return (out, total) if rc == 0 else None


def most_rows(N, chunks, projections, dtype):
    """How many rows there is a launch for."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if dtype == torch.bfloat16:
        return 0 if chunks > 12 else 4 if chunks < 8 or N <= 2 * cus else 8 if chunks == 8 else 6
    return {2: 2, 5: 2, 4: 4, 6: 4, 8: 8 if projections == 2 or -(-N // 16) >= cus else 6}.get(chunks, 0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("projections", [1, 2])
@pytest.mark.parametrize("chunks", range(1, 14))
@pytest.mark.parametrize("M", range(1, 10))
def test_norm_and_product_in_one(M, chunks, projections, dtype):
    """Weight rows that end inside a tile, a tile a workgroup and several, both sides of the lines in weight rows; sizes that have no such launch are refused."""
    k = kern(dtype)
    K = 512 * chunks
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    x, residual, weight = rand((M, K), dtype, 1).cuda(), rand((M, K), dtype, 2).cuda(), rand((K,), dtype, 3).cuda()
    for N in (5, 2 * cus, 2 * cus + 1, 1030, 16 * (cus - 1), 16 * cus - 15, 13001):
        taken = M <= most_rows(N, chunks, projections, dtype)
        assert bool(k.lib.vk_gemm_normed_takes(M, N, K, projections)) == taken, N
        if not taken and N > 5:
            continue
        w = (torch.randn((projections * N, K), generator=torch.Generator("cuda").manual_seed(4), device="cuda") * 0.1).to(dtype)
        got = normed(k, x, residual, weight, 1e-6, w, projections)
        assert (got is not None) == taken, N
        if not taken:
            continue
        total = residual.clone()
        y = k.add_rmsnorm(x, total, weight, 1e-6)
        want = k.gemm(y, w, kernel=4)
        assert torch.equal(got[0], k.swiglu(want) if projections == 2 else want), N
        assert torch.equal(got[1], total)


def test_rows_apart_from_magnitude():
    """A row of zeros, one of the largest values that square within 32 bits and one with an infinity, beside ordinary ones."""
    k = kern(torch.bfloat16)
    K = 2048
    x, residual, weight = rand((4, K), torch.bfloat16, 5).cuda(), rand((4, K), torch.bfloat16, 6).cuda(), rand((K,), torch.bfloat16, 7).cuda()
    x[0], residual[0] = 0, 0
    x[1] *= 1e17
    x[2, 77] = float("inf")
    w = rand((4096, K), torch.bfloat16, 8, 0.1).cuda()
    out, total = normed(k, x, residual, weight, 1e-6, w, 1)
    y = k.add_rmsnorm(x, residual, weight, 1e-6)
    assert torch.equal(out.view(torch.int16), k.gemm(y, w, kernel=4).view(torch.int16)) or torch.equal(out.isnan(), k.gemm(y, w, kernel=4).isnan())
    assert torch.equal(out[[0, 1, 3]], k.gemm(y, w, kernel=4)[[0, 1, 3]]) and torch.equal(total.view(torch.int16), residual.view(torch.int16))


def test_a_negative_eps_is_refused():
    """As the norm by itself refuses it: a NaN in a row whose mean square is smaller would be the only sign of it."""
    k = kern(torch.bfloat16)
    x, residual, weight, w = (rand(s, torch.bfloat16, 9).cuda() for s in ((2, 2048), (2, 2048), (2048,), (4096, 2048)))
    run = k.lib.vk_gemm_normed
    run.argtypes = [P, P, P, P, P, ctypes.c_float, P, I, I, I, ctypes.c_int64, I, P]
    out, total = torch.zeros((2, 4096), dtype=x.dtype, device="cuda"), torch.zeros_like(x)
    rc = run(out.data_ptr(), total.data_ptr(), x.data_ptr(), residual.data_ptr(), weight.data_ptr(), -1e-6, w.data_ptr(), 2, 4096, 2048, 4096, 1,
             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc != 0 and b"eps" in k.lib.vk_last_error() and not out.any() and not total.any()
