"""Decoded rows with four waves a segment: the same bits as the kernels with a wave a segment (plain attention) and as the prompt
rows' kernel at the same position (capped scores, kept keys, windows, sinks)."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, build_cache, kern, rand, run_attention

pytestmark = pytest.mark.gpu

# Keys of a request: one, around a tile of 64, around a segment of 256, a last segment of one tile, and several segments.
LENGTHS = [1, 5, 63, 64, 65, 128, 191, 193, 255, 256, 257, 320, 513, 700]
# The same up to two segments, whose launch folds them itself.
SHORT = [1, 16, 64, 65, 255, 256, 257, 300, 320, 449, 511, 512]


@pytest.mark.parametrize("LENGTHS", [LENGTHS, SHORT], ids=["long", "short"])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,P,window", [(4, 2, 64, 64, 0), (20, 1, 48, 16, 0), (8, 2, 128, 64, 300), (8, 8, 112, 8, 70), (6, 1, 256, 128, 0),
                                               (4, 1, 208, 32, 64)])
def test_plain_rows_agree(LENGTHS, dtype, nq, nkv, d, P, window):
    k = kern(dtype)
    q = [rand((1, nq, d), dtype, 10 + i) for i in range(len(LENGTHS))]
    keys = [rand((n, nkv, d), dtype, 40 + i) for i, n in enumerate(LENGTHS)]
    values = [rand((n, nkv, d), dtype, 70 + i) for i, n in enumerate(LENGTHS)]
    got = {m: run_attention(k, q, keys, values, P, dtype, window=window, poison=float("nan"), seed=m, decode_mode=m, decode_split=m == 7 and max(LENGTHS) > 512) for m in (3, 7, 1)}
    assert not torch.isnan(got[7]).any()
    assert torch.equal(got[7], got[3]) and torch.equal(got[1], got[3])


@pytest.mark.parametrize("LENGTHS", [LENGTHS, SHORT], ids=["long", "short"])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,P,window,keep,cap", [(4, 2, 64, 64, 0, 0, 20.0), (20, 1, 48, 16, 100, 7, 0.0), (8, 2, 128, 64, 300, 16, 20.0),
                                                        (8, 8, 112, 8, 64, 70, 5.0), (6, 1, 256, 128, 0, 0, 0.0)])
def test_capped_rows_agree_with_prompt_rows(LENGTHS, dtype, nq, nkv, d, P, window, keep, cap):
    """The last row of a sequence as a decoded token and as a prompt portion of one row."""
    k = kern(dtype)
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    fn = k.lib.vk_paged_attention_capped
    fn.argtypes = [p] * 5 + [i, p, p, p, i, i, i, p, i, i, i, i, i, i, i, f, f, p, i, p]
    S = len(LENGTHS)
    keys = [rand((n, nkv, d), dtype, 40 + j) for j, n in enumerate(LENGTHS)]
    values = [rand((n, nkv, d), dtype, 70 + j) for j, n in enumerate(LENGTHS)]
    kc, vc, table = (x.cuda() for x in build_cache(keys, values, P, sum(-(-n // P) for n in LENGTHS) + 3, 3, dtype, float("nan")))
    q = torch.cat([rand((1, nq, d), dtype, 10 + j) for j in range(S)]).cuda()
    cu = torch.arange(S + 1, dtype=torch.int32, device="cuda")
    k_len = torch.tensor(LENGTHS, dtype=torch.int32, device="cuda")
    items = torch.stack([torch.arange(S), torch.zeros(S)], 1).to(torch.int32).cuda()
    sinks = torch.linspace(-1, 1, nq, device="cuda")
    nseg = -(-max(LENGTHS) // 256)
    scratch = torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
    out = [torch.zeros_like(q), torch.zeros_like(q)]
    for mode in (0, 1):
        assert fn(out[mode].data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(),
                  items.data_ptr(), S, mode, nseg, scratch.data_ptr(), S, nq, nkv, d, P, window, keep, d ** -0.5, cap, sinks.data_ptr(), 1,
                  torch.cuda.current_stream().cuda_stream) == 0
    assert not torch.isnan(out[1]).any()
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("capped", [False, True])
@pytest.mark.parametrize("nq,nkv,d", [(16, 8, 64), (8, 8, 128), (32, 16, 48)])
def test_many_rows_of_two_segments_and_few(nq, nkv, d, capped, dtype):
    """More workgroups than run at once are folded by a second launch, few fold themselves: the same bits."""
    k, R, P = kern(dtype), 70, 64
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    assert R * nkv > 2 * torch.cuda.get_device_properties(0).multi_processor_count
    lengths = [1 + (37 * j) % 512 for j in range(R - 1)] + [512]
    keys, values = ([rand((n, nkv, d), dtype, s + j) for j, n in enumerate(lengths)] for s in (40, 140))
    kc, vc, table = (x.cuda() for x in build_cache(keys, values, P, sum(-(-n // P) for n in lengths) + 3, 3, dtype, float("nan")))
    q = rand((R, nq, d), dtype, 10).cuda()
    cu, k_len = torch.arange(R + 1, dtype=torch.int32, device="cuda"), torch.tensor(lengths, dtype=torch.int32, device="cuda")
    items = torch.stack([torch.arange(R), torch.zeros(R)], 1).to(torch.int32).cuda()
    scratch = torch.full((k.attn_scratch_floats(R, nq, d, 2),), float("nan"), device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    fn = k.lib.vk_paged_attention_capped if capped else k.lib.vk_paged_attention
    fn.argtypes = [p] * 5 + [i, p, p, p, i, i, i, p, i, i, i, i, i, i] + ([i, f, f, p, i, p] if capped else [f, p])
    tail = (300, 16, d ** -0.5, 20.0, None, 0, stream) if capped else (0, d ** -0.5, stream)
    outs = []
    for n in (R, 7):
        out = torch.full_like(q, float("nan"))
        for at in range(0, R, n):
            assert fn(out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(),
                      items[at:].data_ptr(), n, 1, 2, scratch.data_ptr(), R, nq, nkv, d, P, *tail) == 0
        outs.append(out)
    assert not torch.isnan(outs[0]).any()
    assert torch.equal(*outs)


@pytest.mark.parametrize("LENGTHS", [SHORT, LENGTHS, [1, 300, 1030, 2304, 2305, 2815, 3001]], ids=["short", "long", "longer"])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind,window,keep,block", [("capped", 300, 0, 0), ("capped", 257, 16, 0), ("capped", 2, 600, 0), ("blocked", 0, 0, 200),
                                                    ("blocked", 0, 0, 1024), ("biased", 0, 0, 0), ("biased", 300, 0, 0), ("biased", 513, 70, 0)])
@pytest.mark.parametrize("nq,nkv,d,P", [(4, 2, 64, 64), (20, 1, 112, 8), (6, 1, 208, 128)])
def test_the_variant_s_arguments(LENGTHS, nq, nkv, d, P, kind, window, keep, block, dtype):
    """Windows, kept keys, blocks of positions, biases by distance and a gate a head: a decoded row against the same row as a prompt portion, for requests
    of one segment, of several and of many more than a row sees."""
    k = kern(dtype)
    p, i, l, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
    head = [p] * 5 + [i, p, p, p, i, i, i, p, i, i, i, i, i]
    S = len(LENGTHS)
    keys, values = ([rand((n, nkv, d), dtype, s + j) for j, n in enumerate(LENGTHS)] for s in (40, 70))
    kc, vc, table = (x.cuda() for x in build_cache(keys, values, P, sum(-(-n // P) for n in LENGTHS) + 3, 3, dtype, float("nan")))
    q, gate = rand((S, nq, d), dtype, 10).cuda(), rand((S, nq + 3), dtype, 11).cuda()
    cu = torch.arange(S + 1, dtype=torch.int32, device="cuda")
    k_len = torch.tensor(LENGTHS, dtype=torch.int32, device="cuda")
    items = torch.stack([torch.arange(S), torch.zeros(S)], 1).to(torch.int32).cuda()
    sinks = torch.linspace(-1, 1, nq, device="cuda")
    pad, far = k.lib.vk_attn_rel_pad(), 100
    line = rand((nq, far + 1), torch.float32, 12)                      # the distances far .. 0
    rel = torch.cat([line[:, :1].expand(nq, pad), line, line[:, -1:].expand(nq, pad)], 1).contiguous().cuda()
    nseg = -(-max(LENGTHS) // 256)
    scratch = torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    out = [torch.full_like(q, float("nan")) for _ in range(2)]
    for mode in (0, 1):
        args = (out[mode].data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(),
                items.data_ptr(), S, mode, nseg, scratch.data_ptr(), S, nq, nkv, d, P)
        if kind == "capped":
            fn = k.lib.vk_paged_attention_capped
            fn.argtypes = head + [i, i, f, f, p, i, p]
            rc = fn(*args, window, keep, d ** -0.5, 20.0, sinks.data_ptr(), 1, stream)
        elif kind == "blocked":
            fn = k.lib.vk_paged_attention_blocked
            fn.argtypes = head + [i, f, f, p, i, p]
            rc = fn(*args, block, d ** -0.5, 20.0, sinks.data_ptr(), 1, stream)
        else:
            fn = k.lib.vk_paged_attention_biased
            fn.argtypes = head + [i, i, f, p, i, p, i, i, p, l, p]
            rc = fn(*args, window, keep, d ** -0.5, sinks.data_ptr(), 1, rel.data_ptr(), rel.shape[1], far, gate.data_ptr(), gate.shape[1], stream)
        assert rc == 0
    assert not torch.isnan(out[1]).any()
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("capped", [False, True])
@pytest.mark.parametrize("R,n", [(20, 1000), (70, 1700)])
@pytest.mark.parametrize("nq,nkv,d", [(16, 8, 80), (8, 8, 128), (8, 8, 160), (16, 8, 256)])
def test_many_segments_and_few(nq, nkv, d, R, n, capped, dtype):
    """The number of segments of a launch chooses its kernel: all rows at once and few at a time give the same bits."""
    k, P, nseg = kern(dtype), 64, -(-n // 256)
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    lengths = [1 + (337 * j) % n for j in range(R - 1)] + [n]
    g = torch.Generator(device="cuda").manual_seed(1)
    pages = [-(-m // P) for m in lengths]
    kc, vc = (torch.randn(sum(pages), nkv, P, d, device="cuda", generator=g).to(dtype) for _ in range(2))
    table = torch.zeros(R, max(pages), dtype=torch.int32, device="cuda")
    order = torch.randperm(sum(pages), device="cuda", generator=g).to(torch.int32)
    for r in range(R):
        table[r, :pages[r]] = order[sum(pages[:r]):sum(pages[:r + 1])]
    q = torch.randn(R, nq, d, device="cuda", generator=g).to(dtype)
    cu, k_len = torch.arange(R + 1, dtype=torch.int32, device="cuda"), torch.tensor(lengths, dtype=torch.int32, device="cuda")
    items = torch.stack([torch.arange(R), torch.zeros(R)], 1).to(torch.int32).cuda()
    scratch = torch.full((k.attn_scratch_floats(R, nq, d, nseg),), float("nan"), device="cuda")
    fn = k.lib.vk_paged_attention_capped if capped else k.lib.vk_paged_attention
    fn.argtypes = [p] * 5 + [i, p, p, p, i, i, i, p, i, i, i, i, i, i] + ([i, f, f, p, i, p] if capped else [f, p])
    tail = (0, 0, d ** -0.5, 20.0, None, 0) if capped else (0, d ** -0.5)
    outs = []
    for few in (R, 3):
        out = torch.full_like(q, float("nan"))
        for at in range(0, R, few):
            assert fn(out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(),
                      items[at:].data_ptr(), min(few, R - at), 1, nseg, scratch.data_ptr(), R, nq, nkv, d, P, *tail, torch.cuda.current_stream().cuda_stream) == 0
        outs.append(out)
    assert not torch.isnan(outs[0]).any()
    assert torch.equal(*outs)
