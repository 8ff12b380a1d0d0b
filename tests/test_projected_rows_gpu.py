"""Decoded rows as the projections leave them: the attention that norms, turns and stores them itself gives the bits of vk_qkv_post followed by the attention,
in the output and in the caches."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu
P_, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


def both(dtype, lengths, nq, nkv, d, P, window, norms, turned, missing=(), table_pages=0):
    """(one launch, two launches): outputs and caches; the rows in `missing` have no slot."""
    k = kern(dtype)
    S, pages = len(lengths), [-(-n // P) for n in lengths]
    order = torch.randperm(sum(pages) + 3, generator=torch.Generator().manual_seed(1)).tolist()
    width = max(max(pages), table_pages)
    table = torch.zeros((S, width), dtype=torch.int32)
    for s, n in enumerate(pages):
        table[s, :n] = torch.tensor([order.pop() for _ in range(n)], dtype=torch.int32)
    slots = [-1 if s in missing else int(table[s, (n - 1) // P]) * P + (n - 1) % P for s, n in enumerate(lengths)]
    kc, vc = rand((sum(pages) + 3, nkv, P, d), dtype, 2), rand((sum(pages) + 3, nkv, d, P), dtype, 3)
    for s, n in enumerate(lengths):                          # places that nothing has been written to yet, the row's own among them
        if s not in missing:
            page, at = int(table[s, (n - 1) // P]), (n - 1) % P
            kc[page, :, at:], vc[page, :, :, at:] = float("nan"), float("nan")
    kc, vc, table = kc.cuda(), vc.cuda(), table.cuda()
    qkv = rand((S, (nq + 2 * nkv) * d), dtype, 4).cuda()
    q_w, k_w = (rand((d,), dtype, 5).cuda(), rand((d,), dtype, 6).cuda()) if norms else (None, None)
    cos, sin = (rand((max(lengths), d // 2), dtype, 7).cuda(), rand((max(lengths), d // 2), dtype, 8).cuda()) if turned else (None, None)
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    positions, slot, cu, k_len = dev([n - 1 for n in lengths]), dev(slots), torch.arange(S + 1, dtype=torch.int32, device="cuda"), dev(lengths)
    items = torch.stack([torch.arange(S), torch.zeros(S)], 1).to(torch.int32).cuda()
    nseg = -(-max(width * P, max(lengths)) // 256)
    scratch = torch.full((k.attn_scratch_floats(S, nq, d, nseg),), float("nan"), device="cuda")
    takes, run = k.lib.vk_paged_attention_rows_takes, k.lib.vk_paged_attention_rows
    takes.argtypes = [I] * 6
    run.argtypes = [P_, P_, ctypes.c_int64, P_, P_, P_, P_, F, P_, P_, P_, P_, P_, I, P_, P_, P_, I, I, P_, I, I, I, I, I, F, P_]
    ptr = lambda t: None if t is None else t.data_ptr()
    out, kc1, vc1 = torch.full((S, nq, d), float("nan"), dtype=dtype, device="cuda"), kc.clone(), vc.clone()
    rc = run(ptr(out), ptr(qkv), qkv.shape[1], ptr(kc1), ptr(vc1), ptr(q_w), ptr(k_w), 1e-6, ptr(cos), ptr(sin), ptr(positions), ptr(slot), ptr(table), table.shape[1],
             ptr(cu), ptr(k_len), ptr(items), S, nseg, ptr(scratch), nq, nkv, d, P, window, d ** -0.5, torch.cuda.current_stream().cuda_stream)
    assert (rc == 0) == bool(takes(S, nseg, nq, nkv, d, P))
    if rc:
        return None
    q = k.qkv_post(qkv, nq=nq, nkv=nkv, d=d, q_out=None, k_cache=kc, v_cache=vc, page_size=P, q_w=q_w, k_w=k_w, eps=1e-6, cos=cos, sin=sin, positions=positions, slots=slot)
    scratch.fill_(float("nan"))
    want = k.paged_attention(q, kc, vc, table, cu, k_len, items, mode=1, scale=d ** -0.5, window=window, max_k_len=max(lengths), nseg=nseg, scratch=scratch)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert not torch.isnan(want).any()
    return same(out, want), same(kc1, kc), same(vc1, vc)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,P,window", [(4, 2, 64, 64, 0), (16, 8, 128, 64, 0), (8, 8, 64, 128, 70), (20, 1, 128, 64, 0), (8, 2, 128, 256, 300)])
def test_rows_agree(nq, nkv, d, P, window, dtype):
    """Keys on both sides of the edges of a lane's vector, a tile, a page and a segment; a head a kv head, several, and more than a tile of them."""
    for lengths in ([1, 2, 7, 8, 9, 33, 63, 64, 65, 128], [255, 256, 257, 320, 321, 512], [513, 700, 5]):
        assert both(dtype, lengths, nq, nkv, d, P, window, True, True) == (True, True, True), lengths


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("norms,turned", [(False, True), (True, False), (False, False)])
def test_steps_that_are_left_out(norms, turned, dtype):
    assert both(dtype, [40, 300, 1], 8, 4, 128, 64, 0, norms, turned) == (True, True, True)


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_without_a_slot_and_a_launch_for_longer_requests(dtype):
    """A row that is not stored sees what its cache holds; a recorded step's launch covers more pages than its requests have."""
    assert both(dtype, [40, 64, 300], 8, 4, 64, 64, 0, True, True, missing=(0, 2)) == (True, True, True)
    assert both(dtype, [40, 65, 120], 8, 4, 128, 64, 0, True, True, table_pages=13) == (True, True, True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,norms", [(8, 2, 128, True), (16, 1, 128, True), (17, 1, 64, False), (6, 2, 64, True)])
@pytest.mark.parametrize("window", [0, 40, 70, 300])
def test_waves_without_a_tile(nq, nkv, d, norms, window, dtype):
    """A workgroup a segment in which one to three of the four waves have none: behind the row's own key, and in front of its window."""
    assert both(dtype, [1, 40, 65, 130, 190, 257, 330, 700], nq, nkv, d, 64, window, norms, True, table_pages=13) == (True, True, True)


def test_what_is_not_taken():
    """Heads of other sizes, pages smaller than a tile and more segments than go with four waves each are refused."""
    assert both(torch.bfloat16, [40], 8, 4, 96, 64, 0, True, True) is None
    assert both(torch.bfloat16, [40], 8, 4, 128, 32, 0, True, True) is None
    assert both(torch.bfloat16, [40] * 90, 8, 8, 128, 64, 0, True, True) is None


def test_where_it_is_the_faster_way():
    """One segment a row and several, on both sides of one and two segments a compute unit; never where it is not taken."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for dtype in DTYPES:
        takes, pays = (getattr(kern(dtype).lib, "vk_paged_attention_rows_" + n) for n in ("takes", "preferred"))
        takes.argtypes = pays.argtypes = [I] * 6
        bf16 = dtype == torch.bfloat16
        for nseg in (1, 2, 4):
            for segments in (2 * nseg, cus, cus + 2 * nseg, 2 * cus, 2 * cus + 2 * nseg, 3 * cus):
                rows = segments // (2 * nseg)                # two kv heads
                n = 2 * nseg * rows
                can = [bool(takes(rows, nseg, 4, 2, d, 64)) for d in (64, 128)]
                want = [bf16 or n <= 2 * cus, n <= 2 * cus or nseg > 1 if bf16 else nseg > 1 and n <= cus]
                assert can == [n <= 5 * cus // 2, n <= (5 if bf16 else 12) * cus // 2]
                assert [bool(pays(rows, nseg, 4, 2, d, 64)) for d in (64, 128)] == [a and b for a, b in zip(can, want)], (dtype, nseg, segments)
        assert not pays(4, 2, 4, 2, 96, 64) and not pays(4, 2, 4, 2, 64, 32) and not pays(0, 1, 4, 2, 64, 64)
