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
            want = k.gemm(x[token[at].long()].contiguous(), w[e])
            assert torch.equal(outs[0][at], want) and torch.equal(outs[2][at], want)
            assert torch.equal(outs[1][at], (want.float().clamp(min=0.0) ** 2).to(dtype))
    assert torch.isnan(outs[0][pair < 0]).all()           # nothing is stored there
