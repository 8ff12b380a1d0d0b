"""What one launch does differently for a few tokens and for many gives every token the same bits."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu
P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float


def at(t):
    return None if t is None else t.data_ptr()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,rot_half,norm_d,neighbours", [(128, 64, 128, 0), (128, 32, 96, 0), (256, 128, 256, 1), (80, 40, 80, 1), (64, 1, 0, 0)])
def test_turned_heads_of_many_tokens(d, rot_half, norm_d, neighbours, dtype):
    """A wave's several heads in turn (from 512 tokens on) against a head a wave; rotations of whole heads, of a part, of one pair."""
    k, T, nq, nkv, page = kern(dtype), 515, 5, 2, 16
    width = (nq + 2 * nkv) * d
    x = rand((T, width), dtype, 1).cuda()
    inv = torch.rand(rot_half, generator=torch.Generator().manual_seed(2)).cuda()
    w = (rand((norm_d,), dtype, 3) + 1).cuda() if norm_d else None
    positions = torch.arange(T, dtype=torch.int32, device="cuda") * 7
    slots = torch.arange(T, dtype=torch.int32, device="cuda")
    slots[3] = -1
    fn = k.lib.vk_qkv_post_norm_angles_paired
    fn.argtypes = [P, L, P, P, P, P, P, I, I, F, P, F, I, I, P, P, I, I, I, I, I, P]
    outs = []
    for step in (T, 64):
        q = torch.zeros(T, nq, d, dtype=dtype, device="cuda")
        kc, vc = (torch.zeros(-(-T // page) * nkv * page * d, dtype=dtype, device="cuda") for _ in range(2))
        for t in range(0, T, step):
            n = min(step, T - t)
            assert fn(at(x[t:]), width, at(q[t:]), at(kc), at(vc), at(w), at(w), 0, norm_d, 1e-6, at(inv), 1.25, rot_half, neighbours, at(positions[t:]),
                      at(slots[t:]), n, nq, nkv, d, page, torch.cuda.current_stream().cuda_stream) == 0
        outs.append((q, kc, vc))
    for many, few in zip(*outs):
        assert torch.equal(many, few)
    # The q heads against the equations in 64-bit, from the rounded norms where there are norms.
    h = x[:, :nq * d].reshape(T, nq, d).double()
    if norm_d:
        h = h * torch.rsqrt((h ** 2).sum(-1, keepdim=True) / norm_d + 1e-6)
        h = torch.cat([h[..., :norm_d] * w.double(), torch.zeros_like(h[..., norm_d:])], -1)
    angle = (positions.float()[:, None] * inv).double()[:, None]
    c, s = 1.25 * angle.cos(), 1.25 * angle.sin()
    first, second = (h[..., 0:2 * rot_half:2], h[..., 1:2 * rot_half:2]) if neighbours else (h[..., :rot_half], h[..., rot_half:2 * rot_half])
    a, b = first * c - second * s, second * c + first * s
    turned = torch.stack([a, b], -1).flatten(-2) if neighbours else torch.cat([a, b], -1)
    want = torch.cat([turned, h[..., 2 * rot_half:]], -1)
    # Two roundings to the element type (the norm's, the result's), of values that a rotation by 1.25 mixes in pairs; angles of up to 3,600
    # leave the 32-bit cosines an error of a few units in their last place.
    unit = torch.finfo(dtype).eps
    assert ((outs[0][0].double() - want).abs() <= 3 * unit * (1 + 1.25 * 2 ** 0.5 * h.abs().amax(-1, keepdim=True))).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E,top,groups,keep,kind", [(1, 1, 1, 1, 0), (32, 4, 1, 1, 0), (32, 3, 8, 3, 1), (64, 6, 1, 1, 2), (65, 2, 1, 1, 0), (70, 5, 7, 2, 1)])
def test_routers_of_few_and_many_tokens(E, top, groups, keep, kind, dtype):
    """Choice and plan in one launch (up to 12 or 16 tokens) and in two, an expert a workgroup and four (many tokens and experts); up to 64 experts
    and more.  Every plan is checked: each pair once, in a tile of its expert."""
    k, W = kern(dtype), 224
    h, router = rand((300, W), dtype, 1).cuda(), rand((E, W), dtype, 2, 0.1).cuda()
    correction = rand((E,), dtype, 3, 0.1).cuda() if kind == 1 else None
    fn, most = k.lib.vk_moe_route_plan, k.lib.vk_moe_max_tiles
    fn.argtypes = [P, P, P, P, P, P, I, P, I, I, I, I, I, F, I, I, I, I, F, P, P, P, P, P, I, P]
    most.argtypes = [I, I, I, I]
    whole = None
    for T in (300, 256, 255, 33, 32, 31, 1):
        for tile_rows in (16, 128):
            tiles = most(T, top, E, tile_rows)
            new = lambda *n: torch.full(n, -7, dtype=torch.int32, device="cuda")
            idx, pair, token, pair_row, expert, start = new(T, top), new(tiles * tile_rows), new(tiles * tile_rows), new(T * top), new(tiles), new(E + 1)
            wts = torch.zeros(T, top, device="cuda")
            logits = torch.zeros(T, E, device="cuda")
            assert fn(at(idx), at(wts), at(logits), at(h), at(router), None, 0, at(correction), 0, T, W, E, top, 0.0, kind, groups, keep, 1 if groups > 1 else 0, 2.5,
                      at(pair), at(token), at(pair_row), at(expert), at(start), tile_rows, torch.cuda.current_stream().cuda_stream) == 0
            if whole is None:
                whole = idx, wts, logits
                assert torch.allclose(logits.double(), h.double() @ router.double().T, rtol=0, atol=1e-4)
            for part, all_of_it in zip((idx, wts, logits), whole):
                assert torch.equal(part, all_of_it[:T])
            idx, pair, token, pair_row, expert, start = (v.cpu() for v in (idx.flatten(), pair, token, pair_row, expert, start))
            rows = torch.nonzero(pair >= 0).flatten()
            assert sorted(pair[rows].tolist()) == list(range(T * top))
            assert torch.equal(pair_row[pair[rows].long()].long(), rows)
            assert torch.equal(token[rows], pair[rows] // top) and (token[pair < 0] == 0).all()
            assert torch.equal(expert[rows // tile_rows], idx[pair[rows].long()])
            counts = torch.bincount(idx.long(), minlength=E)
            padded = -(-counts // tile_rows) * tile_rows
            assert start.tolist() == [0] + padded.cumsum(0).tolist()
            assert (expert[start[-1] // tile_rows:] == -1).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E,top,kind", [(32, 4, 0), (32, 5, 1), (64, 1, 0), (64, 8, 2), (72, 4, 0)])
def test_routers_on_both_sides_of_their_lines(E, top, kind, dtype):
    """Choice and plan in one launch or two, one expert a workgroup or four: the choices, weights and logits of a token are the same bits beside any number of
    others, and every plan holds each pair once, in a tile of its expert."""
    k, W = kern(dtype), 224
    many = 600
    h, router = rand((many, W), dtype, 1).cuda(), rand((E, W), dtype, 2, 0.1).cuda()
    fn, most = k.lib.vk_moe_route_plan, k.lib.vk_moe_max_tiles
    fn.argtypes = [P, P, P, P, P, P, I, P, I, I, I, I, I, F, I, I, I, I, F, P, P, P, P, P, I, P]
    most.argtypes = [I, I, I, I]
    whole = None
    for T in (many, 513, 512, 505, 257, 249, 17, 16, 13, 12, 2):
        tiles = most(T, top, E, 16)
        new = lambda *n: torch.full(n, -7, dtype=torch.int32, device="cuda")
        idx, pair, token, pair_row, expert, start = new(T, top), new(tiles * 16), new(tiles * 16), new(T * top), new(tiles), new(E + 1)
        wts, logits = torch.zeros(T, top, device="cuda"), torch.zeros(T, E, device="cuda")
        assert fn(at(idx), at(wts), at(logits), at(h), at(router), None, 0, None, 0, T, W, E, top, 1e-6, kind, 1, 1, 0, 1.0, at(pair), at(token), at(pair_row),
                  at(expert), at(start), 16, torch.cuda.current_stream().cuda_stream) == 0
        if whole is None:
            whole = idx, wts, logits
        for part, all_of_it in zip((idx, wts, logits), whole):
            assert torch.equal(part, all_of_it[:T])
        idx, pair, token, pair_row, expert = (v.cpu() for v in (idx.flatten(), pair, token, pair_row, expert))
        rows = torch.nonzero(pair >= 0).flatten()
        assert sorted(pair[rows].tolist()) == list(range(T * top))
        assert torch.equal(pair_row[pair[rows].long()].long(), rows) and torch.equal(token[rows], pair[rows] // top)
        assert torch.equal(expert[rows // 16], idx[pair[rows].long()])
