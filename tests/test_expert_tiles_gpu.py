"""The experts' products over tiles of 16 rows, by the streaming kernel and by the one for every K: the bits of the plain product."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K", [(16, 32), (40, 96), (333, 512), (64, 544), (200, 1024), (48, 1184), (100, 2560), (96, 3072), (64, 4096), (40, 4608),
                                 (24, 8192), (24, 8224)])
def test_tiles_get_the_plain_product(N, K, dtype):
    """One to five chunks, whole and not, six to eight, nine to sixteen, and more; experts of no, one, 16 and 17 rows."""
    k = kern(dtype)
    counts = [3, 0, 16, 17, 1, 2]
    E, T = len(counts), 20
    g = torch.Generator().manual_seed(2)
    w = rand((E, N, K), dtype, 5, 0.1).cuda()
    x = rand((T, K), dtype, 6).cuda()
    tiles, pairs, tokens, start = [], [], [], [0]
    for e, n in enumerate(counts):
        here = -(-n // 16)
        tiles += [e] * here
        pairs += list(range(len(pairs), len(pairs) + n)) + [-1] * (16 * here - n)
        tokens += torch.randint(0, T, (n,), generator=g).tolist() + [0] * (16 * here - n)
        start.append(len(pairs))
    tiles += [-1, -1]
    pairs, tokens = pairs + [-1] * 32, tokens + [0] * 32
    rows = len(pairs)
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    pair, token, tile, first = dev(pairs), dev(tokens), dev(tiles), dev(start)
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    up, down = k.lib.vk_moe_up_plain, k.lib.vk_moe_down
    act = k.lib.vk_moe_up
    up.argtypes = act.argtypes = [p, l, p, l, p, p, p, p, p, i, i, i, i, i, p]
    down.argtypes = [p, p, l, p, p, p, p, i, i, i, i, i, p]
    stream = torch.cuda.current_stream().cuda_stream
    # The launches cover vk_moe_max_tiles(T, top, E) = (T top + (E - 1 of padding a tile)) / 16 tiles: at least those in use here.
    top = 4
    assert (T * top + min(E, T * top) * 15) // 16 >= len(tiles) - 2
    grid_rows = 16 * ((T * top + min(E, T * top) * 15) // 16)
    pad = lambda v, fill: torch.cat([v, torch.full((max(0, grid_rows - len(v)),), fill, dtype=torch.int32, device="cuda")])
    pair, token = pad(pair, -1), pad(token, 0)
    tile = torch.cat([tile, torch.full((grid_rows // 16,), -1, dtype=torch.int32, device="cuda")])
    gathered = x[token.long()].contiguous()
    gathered[pair < 0] = float("nan")                      # rows without a pair may hold anything
    outs = [torch.full((len(pair), N), float("nan"), dtype=dtype, device="cuda") for _ in range(3)]
    args = (pair.data_ptr(), token.data_ptr(), tile.data_ptr(), first.data_ptr(), T, top, E, N, K, stream)
    assert up(outs[0].data_ptr(), N, x.data_ptr(), K, w.data_ptr(), *args) == 0
    assert act(outs[1].data_ptr(), N, x.data_ptr(), K, w.data_ptr(), *args) == 0
    assert down(outs[2].data_ptr(), gathered.data_ptr(), K, w.data_ptr(), pair.data_ptr(), tile.data_ptr(), first.data_ptr(), T, top, E, N, K, stream) == 0
    for e, n in enumerate(counts):
        if n:
            at = slice(start[e], start[e] + n)
            want = k.gemm(x[token[at].long()].contiguous(), w[e], kernel=3)      # the tile kernel through registers: by size it may be one that brings lines as the experts' does
            assert torch.equal(outs[0][at], want) and torch.equal(outs[2][at], want)
            assert torch.equal(outs[1][at], (want.float().clamp(min=0.0) ** 2).to(dtype))
    assert torch.isnan(outs[0][pair < 0]).all()           # nothing is stored there


@pytest.mark.parametrize("N,K", [(400, 512), (401, 512), (6544, 512), (6545, 512), (400, 1024), (401, 1024), (3264, 1024), (3265, 1024), (192, 2048), (193, 2048), (192, 4096), (193, 4096),
                                 (7, 512), (9, 1024)])
def test_both_sides_of_the_lines(N, K):
    """Ten tiles and 25 and 26, 409 and 410, 204 and 205 groups of 16 features: between which one and two chunks go by a unit a workgroup; 12 and 13 groups, where units are
    more than half of the compute units; features that end inside the first group."""
    test_tiles_get_the_plain_product(N, K, torch.bfloat16)


def offered_plan(counts, offered, top):
    """A plan of `counts` rows an expert, in tiles of 16, as long as the launches of `offered` tokens expect it: pair, token, tile, start."""
    tiles, pairs, start = [], [], [0]
    for e, n in enumerate(counts):
        here = -(-n // 16)
        tiles += [e] * here
        pairs += list(range(len(pairs), len(pairs) + n)) + [-1] * (16 * here - n)
        start.append(len(pairs))
    most = (offered * top + min(len(counts), offered * top) * 15) // 16
    assert len(tiles) <= most
    pairs += [-1] * (16 * most - len(pairs))
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    return dev(pairs), dev(tiles + [-1] * (most - len(tiles))), dev(start)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K", [96, 544, 1184, 1920, 2304, 4640])
def test_an_infinite_weight_gives_infinities(K, dtype):
    """In the last slab of a reduction that ends inside a chunk: the product is infinite with the sign of the row's entry, and no other
    output notices."""
    k, N, top, offered = kern(dtype), 40, 4, 16384
    counts = [5, 16, 2]
    pair, tile, start = offered_plan(counts, offered, top)
    w = rand((len(counts), N, K), dtype, 5, 0.1).cuda()
    x = rand((20, K), dtype, 6).cuda()
    w[1, 7, K - 3] = float("inf")
    token = torch.randint(0, len(x), (len(pair),), generator=torch.Generator().manual_seed(2)).to(torch.int32).cuda()
    rows = x[token.long()].contiguous()
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    up, down = k.lib.vk_moe_up_plain, k.lib.vk_moe_down
    up.argtypes, down.argtypes = [p, l, p, l, p, p, p, p, p, i, i, i, i, i, p], [p, p, l, p, p, p, p, i, i, i, i, i, p]
    outs = [torch.full((len(pair), N), float("nan"), dtype=dtype, device="cuda") for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    sizes = (offered, top, len(counts), N, K, stream)
    assert up(outs[0].data_ptr(), N, x.data_ptr(), K, w.data_ptr(), pair.data_ptr(), token.data_ptr(), tile.data_ptr(), start.data_ptr(), *sizes) == 0
    assert down(outs[1].data_ptr(), rows.data_ptr(), K, w.data_ptr(), pair.data_ptr(), tile.data_ptr(), start.data_ptr(), *sizes) == 0
    at = start.tolist()
    for out in outs:
        for e, n in enumerate(counts):
            got = out[at[e]:at[e] + n].double()
            if e == 1:
                assert torch.equal(got[:, 7], torch.copysign(torch.full_like(got[:, 7], float("inf")), rows[at[e]:at[e] + n, K - 3].double()))
                got[:, 7] = 0.0
            assert torch.isfinite(got).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K", [(4104, 512), (2056, 1024), (1048, 1536), (1048, 2048), (1048, 2560), (264, 4608), (264, 8192), (4104, 480), (2056, 992),
                                 (1048, 1184), (1048, 1920), (1048, 2304)])
def test_workgroups_that_stay_for_several_units(N, K, dtype):
    """More (tile, 16 features) units than the device holds workgroups of the streaming kernel, two to three a workgroup: its window goes on from
    unit to unit, tile to tile and expert to expert, the last features are clamped, and every row in use still gets the plain product."""
    k, top = kern(dtype), 4
    counts = [0, 16, 17, 130, 1, 300, 5, 128]
    used, features = sum(-(-n // 16) for n in counts), -(-N // 16)
    chunks, cus = -(-K // 512), torch.cuda.get_device_properties(0).multi_processor_count
    assert used * features > 2 * cus * (16 // chunks)
    # As many tokens as a launch of this kernel's sizes needs, whichever of its lines applies.
    offered = -(-max(used, -(-12288 // features)) * 16 // top)
    pair, tile, start = offered_plan(counts, offered, top)
    w = torch.randn(len(counts), N, K, device="cuda", generator=torch.Generator(device="cuda").manual_seed(5)).mul_(0.1).to(dtype)
    x = rand((64, K), dtype, 6).cuda()
    token = torch.randint(0, len(x), (len(pair),), generator=torch.Generator().manual_seed(2)).to(torch.int32).cuda()
    token[pair < 0] = 0
    rows = x[token.long()].contiguous()
    rows[pair < 0] = float("nan")                          # rows without a pair may hold anything
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    up, act, down = k.lib.vk_moe_up_plain, k.lib.vk_moe_up, k.lib.vk_moe_down
    up.argtypes = act.argtypes = [p, l, p, l, p, p, p, p, p, i, i, i, i, i, p]
    down.argtypes = [p, p, l, p, p, p, p, i, i, i, i, i, p]
    stream = torch.cuda.current_stream().cuda_stream
    sizes = (offered, top, len(counts), N, K, stream)
    outs = [torch.full((len(pair), N), float("nan"), dtype=dtype, device="cuda") for _ in range(3)]
    for fn, out in ((up, outs[0]), (act, outs[1])):
        assert fn(out.data_ptr(), N, x.data_ptr(), K, w.data_ptr(), pair.data_ptr(), token.data_ptr(), tile.data_ptr(), start.data_ptr(), *sizes) == 0
    assert down(outs[2].data_ptr(), rows.data_ptr(), K, w.data_ptr(), pair.data_ptr(), tile.data_ptr(), start.data_ptr(), *sizes) == 0
    at = start.tolist()
    for e, n in enumerate(counts):
        if n:
            here = slice(at[e], at[e] + n)
            want = k.gemm(rows[here].contiguous(), w[e], kernel=3)
            assert torch.equal(outs[0][here], want) and torch.equal(outs[2][here], want)
            assert torch.equal(outs[1][here], (want.float().clamp(min=0.0) ** 2).to(dtype))
    assert all(torch.isnan(out[pair < 0]).all() for out in outs)          # nothing is stored there
