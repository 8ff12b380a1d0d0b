"""Decoded attention without a list of items: row i is all that sequence i brings.  The same bits as with the list that says so."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, build_cache, kern, rand

pytestmark = pytest.mark.gpu
P_, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
LISTS = P_, P_, P_, I, I, I, P_, I, I, I, I, I
# Around a lane's vector, a tile and a segment; up to two segments, up to four, and more (the fold fetches four at a time).
LENGTHS = {"two": [1, 7, 8, 33, 64, 65, 255, 256, 257, 512], "four": [5, 300, 513, 1024], "nine": [64, 700, 2100]}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("nq,nkv,d,P,window,keep,cap", [(8, 2, 128, 64, 0, 0, 20.0), (20, 1, 64, 128, 100, 7, 0.0), (6, 1, 256, 64, 300, 70, 5.0), (4, 4, 48, 16, 64, 0, 0.0)])
def test_lists_and_none_agree(nq, nkv, d, P, window, keep, cap, lengths, dtype):
    k, n = kern(dtype), LENGTHS[lengths]
    S, lib, stream = len(n), kern(dtype).lib, torch.cuda.current_stream().cuda_stream
    keys, values = ([rand((m, nkv, d), dtype, s + j) for j, m in enumerate(n)] for s in (40, 140))
    kc, vc, table = (x.cuda() for x in build_cache(keys, values, P, sum(-(-m // P) for m in n) + 3, 3, dtype, float("nan")))
    q = torch.cat([rand((1, nq, d), dtype, 10 + j) for j in range(S)]).cuda()
    cu, k_len = torch.arange(S + 1, dtype=torch.int32, device="cuda"), torch.tensor(n, dtype=torch.int32, device="cuda")
    items = torch.stack([torch.arange(S), torch.zeros(S)], 1).to(torch.int32).cuda()
    sinks = torch.linspace(-1, 1, nq, device="cuda")
    nseg = -(-max(n) // 256)

    def both(fn, mode, *rest):
        fn.argtypes = [P_] * 5 + [I, *LISTS, *(t for t, _ in rest), P_]
        outs = []
        for listed in (True, False):
            out, scratch = torch.full_like(q, float("nan")), torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
            assert fn(out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr() if listed else None, k_len.data_ptr(),
                      items.data_ptr() if listed else None, S, mode, nseg, scratch.data_ptr(), S, nq, nkv, d, P, *(v for _, v in rest), stream) == 0
            outs.append(out)
        assert not torch.isnan(outs[0]).any() and torch.equal(*outs)

    for mode in (1, 3, 4, 7):
        both(lib.vk_paged_attention, mode, (I, window), (F, d ** -0.5))
    both(lib.vk_paged_attention_capped, 1, (I, window), (I, keep), (F, d ** -0.5), (F, cap), (P_, sinks.data_ptr()), (I, 1))
    assert lib.vk_paged_attention(q.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(),
                                  None, S, 0, nseg, None, S, nq, nkv, d, P, window, d ** -0.5, stream) != 0       # prompt rows need theirs


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d", [(16, 8, 128), (20, 1, 128), (16, 1, 64), (8, 8, 64)])
def test_projected_rows_without_a_list(nq, nkv, d, dtype):
    """Kv heads with one q head, several, sixteen (the key's row is the seventeenth) and more."""
    k, P = kern(dtype), 64
    lib, stream = k.lib, torch.cuda.current_stream().cuda_stream
    for n in ([1, 30, 64, 65, 256], [257, 511, 3], [700]):
        S, pages = len(n), [-(-m // P) for m in n]
        table, at = torch.zeros((S, max(pages)), dtype=torch.int32), 0
        for s, m in enumerate(pages):
            table[s, :m] = torch.arange(at, at + m, dtype=torch.int32)
            at += m
        dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
        slots, positions, k_len = dev([int(table[s, (m - 1) // P]) * P + (m - 1) % P for s, m in enumerate(n)]), dev([m - 1 for m in n]), dev(n)
        cu, items, table = dev(list(range(S + 1))), dev([[s, 0] for s in range(S)]), table.cuda()
        kc, vc, qkv = rand((at, nkv, P, d), dtype, 2).cuda(), rand((at, nkv, d, P), dtype, 3).cuda(), rand((S, (nq + 2 * nkv) * d), dtype, 4).cuda()
        w, cos, sin = rand((2, d), dtype, 5).cuda(), rand((max(n), d // 2), dtype, 7).cuda(), rand((max(n), d // 2), dtype, 8).cuda()
        nseg = -(-max(n) // 256)
        run = lib.vk_paged_attention_rows
        run.argtypes = [P_, P_, ctypes.c_int64, P_, P_, P_, P_, F, P_, P_, P_, P_, P_, I, P_, P_, P_, I, I, P_, I, I, I, I, I, F, P_]
        got = []
        for listed in (True, False):
            out, kc1, vc1 = torch.full((S, nq, d), float("nan"), dtype=dtype, device="cuda"), kc.clone(), vc.clone()
            scratch = torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
            assert run(out.data_ptr(), qkv.data_ptr(), qkv.shape[1], kc1.data_ptr(), vc1.data_ptr(), w[0].data_ptr(), w[1].data_ptr(), 1e-6, cos.data_ptr(), sin.data_ptr(),
                       positions.data_ptr(), slots.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr() if listed else None, k_len.data_ptr(),
                       items.data_ptr() if listed else None, S, nseg, scratch.data_ptr(), nq, nkv, d, P, 0, d ** -0.5, stream) == 0
            got.append((out, kc1, vc1))
        assert not torch.isnan(got[0][0]).any() and all(torch.equal(a, b) for a, b in zip(*got)), n


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [[0, 5, 300], [130, 0, 700], [64, 0, 2100, 0]], ids=["two", "three", "nine"])
@pytest.mark.parametrize("nq,nkv,d,P,window,keep", [(8, 2, 128, 64, 0, 0), (4, 4, 48, 16, 64, 7), (6, 1, 256, 64, 300, 70)])
def test_a_sequence_without_keys(nq, nkv, d, P, window, keep, n, dtype):
    """Its row is zeros, whatever its pages hold, and the other rows are what they are beside sequences with a key."""
    k, S = kern(dtype), len(n)
    lib, stream, nseg = k.lib, torch.cuda.current_stream().cuda_stream, -(-max(n) // 256)
    keys, values = ([rand((m, nkv, d), dtype, s + j) for j, m in enumerate(n)] for s in (40, 140))
    kc, vc, table = (x.cuda() for x in build_cache(keys, values, P, sum(-(-m // P) for m in n) + 3, 3, dtype, float("nan")))
    q = torch.cat([rand((1, nq, d), dtype, 10 + j) for j in range(S)]).cuda()
    cu, items = torch.arange(S + 1, dtype=torch.int32, device="cuda"), torch.stack([torch.arange(S), torch.zeros(S)], 1).to(torch.int32).cuda()
    sinks, empty = torch.linspace(-1, 1, nq, device="cuda"), torch.tensor([m == 0 for m in n], device="cuda")
    plain, capped = lib.vk_paged_attention, lib.vk_paged_attention_capped
    plain.argtypes, capped.argtypes = [P_] * 5 + [I, *LISTS, I, F, P_], [P_] * 5 + [I, *LISTS, I, I, F, F, P_, I, P_]

    def run(fn, lengths, listed, mode, *rest):
        out, scratch = torch.full_like(q, float("nan")), torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
        k_len = torch.tensor(lengths, dtype=torch.int32, device="cuda")
        assert fn(out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr() if listed else None, k_len.data_ptr(),
                  items.data_ptr() if listed else None, S, mode, nseg, scratch.data_ptr(), S, nq, nkv, d, P, *rest, stream) == 0
        return out

    calls = [(plain, mode, window, d ** -0.5) for mode in (1, 3, 4, 5, 7)] + [(capped, 1, window, keep, d ** -0.5, 5.0, sinks.data_ptr(), 1)]
    for fn, *rest in calls:
        for listed in (True, False):
            out, beside = run(fn, n, listed, *rest), run(fn, [max(m, 1) for m in n], listed, *rest)
            assert not out[empty].any() and torch.equal(out[~empty], beside[~empty]) and not torch.isnan(out[~empty]).any(), rest


@pytest.mark.parametrize("dtype", DTYPES)
def test_lists_that_are_refused(dtype):
    """Prompt rows without items, rows without items that are not all of them, items without their sequences' first rows."""
    k, P, d = kern(dtype), 64, 64
    lib, stream = k.lib, torch.cuda.current_stream().cuda_stream
    cache, q, scratch = torch.zeros(2, 1, P, d, dtype=dtype, device="cuda"), torch.zeros(2, 3, d, dtype=dtype, device="cuda"), torch.zeros(4096, device="cuda")
    ints = torch.ones(2, 2, dtype=torch.int32, device="cuda")
    plain, capped, rows = lib.vk_paged_attention, lib.vk_paged_attention_capped, lib.vk_paged_attention_rows
    plain.argtypes, capped.argtypes = [P_] * 5 + [I, *LISTS, I, F, P_], [P_] * 5 + [I, *LISTS, I, I, F, F, P_, I, P_]
    for fn, rest in ((plain, (0, 1.0)), (capped, (0, 0, 1.0, 0.0, None, 0))):
        for listed, cu, n_items, mode in ((False, True, 2, 0), (False, False, 1, 1), (False, False, 3, 1), (True, False, 2, 1), (True, False, 2, 0)):
            assert fn(q.data_ptr(), q.data_ptr(), cache.data_ptr(), cache.data_ptr(), ints.data_ptr(), 2, ints.data_ptr() if cu else None, ints.data_ptr(),
                      ints.data_ptr() if listed else None, n_items, mode, 1, scratch.data_ptr(), 2, 3, 1, d, P, *rest, stream) != 0, (listed, cu, n_items, mode)
    rows.argtypes = [P_, P_, ctypes.c_int64, P_, P_, P_, P_, F, P_, P_, P_, P_, P_, I, P_, P_, P_, I, I, P_, I, I, I, I, I, F, P_]
    assert rows(q.data_ptr(), q.data_ptr(), 5 * d, cache.data_ptr(), cache.data_ptr(), None, None, 1e-6, None, None, ints.data_ptr(), ints.data_ptr(), ints.data_ptr(), 2,
                None, ints.data_ptr(), ints.data_ptr(), 1, 1, scratch.data_ptr(), 3, 1, d, P, 0, 1.0, stream) != 0
