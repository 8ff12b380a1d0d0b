"""Prompt rows of the variant (capped scores, sinks, windows that keep the first keys): tiles shared in LDS against the kernel for every shape, and both against
the same attention in 64 bits.  Pages that lie between the kept keys and the window have been given back: they hold NaN."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, build_cache, kern, rand

pytestmark = pytest.mark.gpu
P_, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
ITEM_ROWS = 128
FEW = [(150, 150), (40, 700)]                                                                      # (rows, keys) of a request
MANY = [(300, 300), (129, 641), (2, 64), (33, 289), (128, 128), (97, 1000), (31, 95), (64, 576), (257, 1300)]


def wanted(q, keys, values, window, keep, cap, sinks):
    """In 64 bits; q [rows, nq, d], keys and values [n, nkv, d]."""
    rows, nq, d = q.shape
    n, group = keys.shape[0], nq // keys.shape[1]
    pos, key = torch.arange(n - rows, n)[:, None], torch.arange(n)[None]
    seen = (key <= pos) & ((key > pos - window) | (key < keep) if window else True)
    kk, vv = (x.double().repeat_interleave(group, 1).transpose(0, 1).contiguous() for x in (keys, values))
    s = q.double().transpose(0, 1).contiguous() @ kk.transpose(1, 2).contiguous() * d ** -0.5
    s = cap * torch.tanh(s / cap) if cap else s
    s = torch.where(seen, s, -torch.inf)
    top = s.amax(-1, keepdim=True)
    e = torch.exp(s - top)
    return ((e @ vv) / (e.sum(-1, keepdim=True) + torch.exp(sinks.double()[:, None, None] - top))).transpose(0, 1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shapes", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("window,keep,cap", [(0, 0, 5.0), (70, 0, 0.0), (64, 64, 0.0), (100, 7, 20.0), (130, 200, 5.0), (1, 1, 0.0), (300, 65, 0.0)])
@pytest.mark.parametrize("nq,nkv,d", [(4, 2, 64), (6, 1, 128), (8, 2, 192), (32, 1, 256)])
def test_shared_tiles_the_general_kernel_and_64_bits(nq, nkv, d, window, keep, cap, shapes, dtype):
    """Kept keys that end at a tile's edge, inside it and in the window; tiles seen whole among them; heads of 256 in a few items and in many."""
    k, total = kern(dtype), sum(r for r, _ in shapes)
    q, keys, values = ([rand(size, dtype, seed + j) for j, size in enumerate(sizes)] for seed, sizes in
                       ((10, [(r, nq, d) for r, _ in shapes]), (40, [(n, nkv, d) for _, n in shapes]), (70, [(n, nkv, d) for _, n in shapes])))
    sinks = torch.linspace(-1, 1, nq)
    rows, starts, at = torch.cat(q).cuda(), [0], 0
    for r, _ in shapes:
        at += r
        starts.append(at)
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    cu, k_len, items = dev(starts), dev([n for _, n in shapes]), dev([[s, o] for s, (r, _) in enumerate(shapes) for o in range(0, r, ITEM_ROWS)])
    sinks_gpu = sinks.cuda()
    fn = k.lib.vk_paged_attention_capped
    fn.argtypes = [P_] * 5 + [I, P_, P_, P_, I, I, I, P_, I, I, I, I, I, I, I, F, F, P_, I, P_]
    got = []
    for P in (64, 16):                                  # pages smaller than a tile go to the kernel for every shape
        assert P == 64 or not k.lib.vk_attn_prefill_shares_tiles(d, P)
        kc, vc, table = build_cache(keys, values, P, sum(-(-n // P) for _, n in shapes) + 3, 3, dtype, float("nan"))
        for s, (r, n) in enumerate(shapes):
            first = max(0, n - r - window + 1) if window else 0
            for page in range(-(-n // P)):
                if page * P >= keep and (page + 1) * P <= first:
                    table[s, page] = table[0, -1]
        kc, vc, table, out = kc.cuda(), vc.cuda(), table.cuda(), torch.full_like(rows, float("nan"))
        assert fn(out.data_ptr(), rows.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], cu.data_ptr(), k_len.data_ptr(), items.data_ptr(),
                  len(items), 0, 0, None, total, nq, nkv, d, P, window, keep, d ** -0.5, cap, sinks_gpu.data_ptr(), 1, torch.cuda.current_stream().cuda_stream) == 0
        got.append(out.cpu())
    assert torch.equal(*got)
    # 32-bit sums of n products: n / 2^24 of the largest terms, a dozen units at most here; then the result's own rounding.
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    for s, (r, _) in enumerate(shapes):
        want, have = wanted(q[s], keys[s], values[s], window, keep, cap, sinks), got[0][starts[s]:starts[s + 1]].double()
        assert ((have - want).abs() <= unit * want.abs() + 4e-5).all()
