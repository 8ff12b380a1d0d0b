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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,lda", [(256, 512, 512), (96, 1024, 1088), (1100, 512, 520), (300, 192, 192)])
def test_named_rows_are_as_their_copy(N, K, lda, dtype):
    """Rows that a table names out of order, several times and never, against their copy in the product's order; rows further apart than
    they are long; K of whole chunks and not; few workgroups and many."""
    k = kern(dtype)
    g = torch.Generator().manual_seed(3)
    for experts, T in ((2, 1), (40, 333)):
        w = rand((experts, N, K), dtype, 5, 0.1).cuda()
        x = rand((T, lda), dtype, 6).cuda()
        counts = torch.randint(0, 130, (experts,), generator=g).tolist()
        blocks = [e for e, n in enumerate(counts) for _ in range(-(-n // 128))] + [-1]
        M = 128 * len(blocks)
        pairs, at = torch.full((M,), -1, dtype=torch.int32), 0
        for n in counts:
            pairs[at:at + n] = torch.arange(n, dtype=torch.int32)
            at += 128 * (-(-n // 128))
        named = torch.randint(0, T, (M,), generator=g, dtype=torch.int32)
        copy = x[named.long().cuda()].contiguous()
        which, row_pair, row = (torch.as_tensor(v, dtype=torch.int32).cuda() for v in (blocks, pairs, named))
        p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
        fn = k.lib.vk_gemm_grouped_rows
        fn.argtypes = [p, p, p, i, i, i, l, l, p, l, p, p, i, i, p]
        stream = torch.cuda.current_stream().cuda_stream
        outs = [torch.zeros(M, N, dtype=dtype, device="cuda") for _ in range(2)]
        for out, act, rows in ((outs[0], copy, None), (outs[1], x, row.data_ptr())):
            assert fn(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, lda, N, which.data_ptr(), N * K, row_pair.data_ptr(), rows, T, 0, stream) == 0
        assert torch.equal(*outs)
        # More bytes than the offsets reach are refused.
        assert fn(outs[0].data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, lda, N, which.data_ptr(), N * K, None, row.data_ptr(), 1 << 30, 0, stream) != 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,activation", [(96, 1024, 1), (256, 512, 0), (1100, 512, 0), (2048, 512, 0), (4200, 512, 1), (4400, 512, 0), (4400, 192, 0)])
def test_workgroups_of_both_widths(N, K, activation, dtype):
    """The number of matrices, said or not, chooses between workgroups of 256 and of 128 weight rows: the same bits, rows named and copied, idle halves
    and none.  More than 4,096 weight rows are walked in two bands of column blocks; they end inside a workgroup's tile."""
    k = kern(dtype)
    g = torch.Generator().manual_seed(3)
    counts = [1, 63, 64, 65, 128, 0, 129, 200]
    w = rand((len(counts), N, K), dtype, 5, 0.1).cuda()
    x = rand((77, K), dtype, 6).cuda()
    blocks, pairs = [], []
    for e, n in enumerate(counts):
        here = -(-n // 128)
        blocks += [e] * here
        pairs += list(range(n)) + [-1] * (128 * here - n)
    blocks, pairs = blocks + [-1], pairs + [-1] * 128
    M = len(pairs)
    named = torch.randint(0, len(x), (M,), generator=g, dtype=torch.int32)
    copy = x[named.long().cuda()].contiguous()
    which, row_pair, row = (torch.as_tensor(v, dtype=torch.int32).cuda() for v in (blocks, pairs, named))
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_gemm_grouped_experts
    fn.argtypes = [p, p, p, i, i, i, l, l, p, l, i, p, p, i, i, p]
    stream = torch.cuda.current_stream().cuda_stream
    for matrices in (0, len(counts)):
        for act, rows in ((copy, None), (x, row.data_ptr())):
            for given in (None, row_pair.data_ptr()):
                out = torch.zeros(M, N, dtype=dtype, device="cuda")
                assert fn(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, K, N, which.data_ptr(), N * K, matrices, given, rows, len(x), activation,
                          stream) == 0
                at = 0
                for e, n in enumerate(counts):
                    if n:
                        want = k.gemm(copy[at:at + n], w[e])
                        if activation:
                            want = (want.float().clamp(min=0.0) ** 2).to(dtype)
                        assert torch.equal(out[at:at + n], want)
                    at += 128 * (-(-n // 128))
                assert (out[M - 128:] == 0).all()          # the block that is not in use
