"""The tile product with blocks of rows that are half or wholly empty: the rows in use get the bits of the plain product."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,activation", [(256, 512, 0), (96, 1024, 1), (1100, 512, 0), (300, 192, 0)])
def test_rows_in_use_get_the_plain_product(N, K, activation, dtype):
    """Groups of 1 to 200 rows in blocks of 128 (up to 64 rows in the last one leave half of it idle), one group without rows, and a
    block beyond the last; weight rows that end inside a workgroup's tile; K of whole chunks and not."""
    k = kern(dtype)
    counts = [1, 63, 64, 65, 128, 0, 129, 200]
    w = rand((len(counts), N, K), dtype, 5, 0.1).cuda()
    blocks, pairs, rows = [], [], []
    for e, n in enumerate(counts):
        here = -(-n // 128)
        blocks += [e] * here
        pairs += list(range(n)) + [-1] * (128 * here - n)
        rows.append(n)
    blocks, pairs = blocks + [-1], pairs + [-1] * 128
    M = len(pairs)
    act = rand((M, K), dtype, 6).cuda()
    out = torch.zeros(M, N, dtype=dtype, device="cuda")
    which, row_pair = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in (blocks, pairs))
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_gemm_grouped_act
    fn.argtypes = [p, p, p, i, i, i, l, l, p, l, p, i, p]
    for given in (None, row_pair.data_ptr()):
        out.zero_()
        assert fn(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, K, N, which.data_ptr(), N * K, given, activation,
                  torch.cuda.current_stream().cuda_stream) == 0
        at = 0
        for e, n in enumerate(rows):
            if n:
                want = k.gemm(act[at:at + n].contiguous(), w[e])
                if activation:
                    want = (want.float().clamp(min=0.0) ** 2).to(dtype)
                assert torch.equal(out[at:at + n], want)
            at += 128 * (-(-n // 128))
