"""The experts' product by a plan's order: the plain product's bits for every row that has a pair, the gated activation in its epilogue, and the order itself."""
import ctypes

import pytest
import torch
from test_kernels_gpu import kern, rand

pytestmark = pytest.mark.gpu
P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
PART = 192                              # rows of a part, at most
BF16 = torch.bfloat16
# Around the six heights of a part, more than one part, no rows at all; more matrices than a wave has lanes.
COUNTS = {"heights": [1, 32, 33, 64, 96, 97, 0, 128, 160, 161, 192], "parts": [193, 0, 384, 385, 700, 2], "many": [i % 5 * 20 for i in range(70)]}


def stream():
    return torch.cuda.current_stream().cuda_stream


def layout(counts):
    """First rows of the matrices' runs (whole blocks of 128) and the order of a plan for them, the matrices in sequence."""
    starts, at, order, before = [], 0, [], 0
    for e, n in enumerate(counts):
        starts.append(at)
        if n:
            order.append([before, at, n, e])
        before += -(-n // PART)
        at += -(-n // 128) * 128
    order += [[before, 0, 0, 0]] * (len(counts) - len(order))
    return starts, at + 128, torch.tensor(order, dtype=torch.int32)


@pytest.mark.parametrize("which", COUNTS)
@pytest.mark.parametrize("N,K,lda,activation", [(256, 512, 512, 0), (300, 1024, 1032, 1), (1101, 512, 520, 0)])
def test_rows_of_an_order_get_the_plain_product(which, N, K, lda, activation):
    """Rows named and as they lie, columns that end inside a tile and such as are no multiple of four, one chunk and two."""
    k, counts = kern(BF16), COUNTS[which]
    starts, M, order = layout(counts)
    order = order.cuda()
    w = rand((len(counts), N, K), BF16, 5, 0.1).cuda()
    x = rand((333, lda), BF16, 6).cuda()
    named = torch.randint(0, len(x), (M,), generator=torch.Generator().manual_seed(3), dtype=torch.int32)
    copy, named = x[named.long().cuda()].contiguous(), named.cuda()
    fn = k.lib.vk_gemm_experts
    fn.argtypes = [P, P, P, I, I, I, L, L, P, I, L, P, I, I, P]
    for act, rows in ((copy, None), (x, named.data_ptr())):
        out = torch.full((M, N), 7.0, dtype=BF16, device="cuda")
        assert fn(out.data_ptr(), act.data_ptr(), w.data_ptr(), M, N, K, lda, N, order.data_ptr(), len(counts), N * K, rows, len(x), activation, stream()) == 0
        held = torch.zeros(M, dtype=torch.bool)
        for e, (at, n) in enumerate(zip(starts, counts)):
            if n:
                want = k.gemm(copy[at:at + n, :K].contiguous(), w[e])
                if activation:
                    want = (want.float().clamp(min=0.0) ** 2).to(BF16)
                assert torch.equal(out[at:at + n], want)
                held[at:at + n] = True
        assert (out[~held.cuda()] == 7.0).all()


@pytest.mark.parametrize("which", COUNTS)
@pytest.mark.parametrize("width,K,limit,weighed", [(128, 512, 7.0, False), (200, 512, float("inf"), True), (264, 1024, 0.5, True)])
def test_gated_activation_as_a_pass_of_its_own(which, width, K, limit, weighed):
    """vk_gemm_experts_glu against the product, then vk_moe_glu or vk_moe_glu_weighed: the same bits."""
    k, counts = kern(BF16), COUNTS[which]
    starts, M, order = layout(counts)
    order = order.cuda()
    w = rand((len(counts), 2 * width, K), BF16, 5, 0.1).cuda()
    x = rand((M, K), BF16, 6).cuda()
    pair = torch.full((M,), -1, dtype=torch.int32)
    for at, n in zip(starts, counts):
        pair[at:at + n] = torch.arange(at, at + n, dtype=torch.int32)
    wts = torch.rand(M, generator=torch.Generator().manual_seed(2)).cuda()
    held, pair = pair.cuda() >= 0, pair.cuda()
    args = (pair.data_ptr(), wts.data_ptr()) if weighed else (None, None)
    fn = k.lib.vk_gemm_experts_glu
    fn.argtypes = [P, P, P, I, I, I, L, L, P, I, L, P, I, F, F, F, P, P, P]
    out = torch.zeros(M, width, dtype=BF16, device="cuda")
    assert fn(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, width, K, K, width, order.data_ptr(), len(counts), 2 * width * K, None, 0, limit, 1.702, 1.0, *args, stream()) == 0
    both = torch.zeros(M, 2 * width, dtype=BF16, device="cuda")
    for e, (at, n) in enumerate(zip(starts, counts)):
        if n:
            both[at:at + n] = k.gemm(x[at:at + n], w[e])
    want = torch.zeros_like(out)
    glu = k.lib.vk_moe_glu_weighed if weighed else k.lib.vk_moe_glu
    glu.argtypes = [P, P, L, I, F, F, F] + ([P, P] if weighed else []) + [P]
    assert glu(want.data_ptr(), both.data_ptr(), M, width, limit, 1.702, 1.0, *(args if weighed else ()), stream()) == 0
    assert torch.equal(out[held], want[held])


def test_what_is_refused():
    k = kern(BF16)
    fn = k.lib.vk_gemm_experts
    fn.argtypes = [P, P, P, I, I, I, L, L, P, I, L, P, I, I, P]
    x, w, order = torch.zeros(128, 512, dtype=BF16, device="cuda"), torch.zeros(1, 256, 512, dtype=BF16, device="cuda"), torch.zeros(4, dtype=torch.int32, device="cuda")
    good = [x.data_ptr(), x.data_ptr(), w.data_ptr(), 128, 256, 512, 512, 256, order.data_ptr(), 1, 256 * 512, None, 0, 0, stream()]
    for place, bad in ((3, 100), (4, 255), (5, 640), (6, 500), (7, 255), (8, None), (9, 0), (13, 2)):
        assert fn(*good[:place], bad, *good[place + 1:]) != 0
    assert fn(*good[:11], order.data_ptr(), 1 << 30, *good[13:]) != 0          # named rows beyond what 31 bits reach


class Plan:
    """vk_moe_route_plan_ordered over tokens h, with or without a router bias."""

    def __init__(self, k, h, router, top, bias=None):
        T, E = len(h), len(router)
        most = k.lib.vk_moe_max_tiles
        most.argtypes = [I, I, I, I]
        self.tiles = most(T, top, E, 128)
        new = lambda *n: torch.full(n, -7, dtype=torch.int32, device="cuda")
        self.idx, self.pair, self.token, self.pair_row = new(T, top), new(self.tiles * 128), new(self.tiles * 128), new(T * top)
        self.expert, self.start, self.order = new(self.tiles), new(E + 1), new(E, 4)
        self.wts, logits = torch.zeros(T, top, device="cuda"), torch.zeros(T, E, device="cuda")
        fn = k.lib.vk_moe_route_plan_ordered
        fn.argtypes = [P, P, P, P, P, P, I, P, I, I, I, I, I, F, I, I, I, I, F, P, P, P, P, P, I, P, P]
        assert fn(self.idx.data_ptr(), self.wts.data_ptr(), logits.data_ptr(), h.data_ptr(), router.data_ptr(), bias.data_ptr() if bias is not None else None, 1, None, 0, T,
                  h.shape[1], E, top, 0.0, 0, 1, 1, 0, 1.0, self.pair.data_ptr(), self.token.data_ptr(), self.pair_row.data_ptr(), self.expert.data_ptr(),
                  self.start.data_ptr(), 128, self.order.data_ptr(), stream()) == 0
        self.counts = torch.bincount(self.idx.flatten().long().cpu(), minlength=E).tolist()


@pytest.mark.parametrize("form", ["gated", "weighed", "squared"])
@pytest.mark.parametrize("E,T,top,W,width", [(32, 640, 3, 1024, 1024), (70, 900, 4, 1024, 512), (5, 3000, 2, 512, 1024)])
def test_experts_of_a_plan(E, T, top, W, width, form):
    """Tokens through a plan, both products and what stands between them: the same bits as by the plan's blocks, and the experts' formula in 32 bits.  The router's bias
    leaves experts without rows and gives others several parts, so that the order is not the experts' own."""
    k = kern(BF16)
    x, router = rand((T, W), BF16, 1).cuda(), rand((E, W), BF16, 2, W ** -0.5).cuda()
    bias = (torch.randn(E, generator=torch.Generator().manual_seed(4)) * 3).cuda()
    p = Plan(k, x, router, top, bias)
    assert max(p.counts) > PART and (E < 10 or min(p.counts) == 0)
    listed = [e for _, _, rows, e in p.order.tolist() if rows]
    assert E > 64 or listed != sorted(listed)
    both = 1 if form == "squared" else 2
    up, down = rand((E, both * width, W), BF16, 5, W ** -0.5).cuda(), rand((E, W, width), BF16, 6, width ** -0.5).cuda()
    M, held = p.tiles * 128, p.pair >= 0
    limit, slope, shift = 1.5, 1.702, 1.0
    weighed = (p.pair.data_ptr(), p.wts.data_ptr()) if form == "weighed" else (None, None)
    blocks, parts = k.lib.vk_gemm_grouped_experts, k.lib.vk_gemm_experts
    blocks.argtypes = [P, P, P, I, I, I, L, L, P, L, I, P, P, I, I, P]
    parts.argtypes = [P, P, P, I, I, I, L, L, P, I, L, P, I, I, P]
    empty = lambda n: torch.full((M, n), float("nan"), dtype=BF16, device="cuda")       # as memory that nobody has written
    relu = int(form == "squared")

    act, first = empty(width), empty(both * width)
    assert blocks(first.data_ptr(), x.data_ptr(), up.data_ptr(), M, both * width, W, W, both * width, p.expert.data_ptr(), both * width * W, E, p.pair.data_ptr(),
                  p.token.data_ptr(), T, relu, stream()) == 0
    if form == "squared":
        act = first
    else:
        glu = k.lib.vk_moe_glu_weighed if form == "weighed" else k.lib.vk_moe_glu
        glu.argtypes = [P, P, L, I, F, F, F] + ([P, P] if form == "weighed" else []) + [P]
        assert glu(act.data_ptr(), first.data_ptr(), M, width, limit, slope, shift, *(weighed if form == "weighed" else ()), stream()) == 0
    want = empty(W)
    assert blocks(want.data_ptr(), act.data_ptr(), down.data_ptr(), M, W, width, width, W, p.expert.data_ptr(), W * width, E, p.pair.data_ptr(), None, 0, 0, stream()) == 0

    gated, got = empty(width), empty(W)
    if form == "squared":
        assert parts(gated.data_ptr(), x.data_ptr(), up.data_ptr(), M, width, W, W, width, p.order.data_ptr(), E, width * W, p.token.data_ptr(), T, 1, stream()) == 0
    else:
        fn = k.lib.vk_gemm_experts_glu
        fn.argtypes = [P, P, P, I, I, I, L, L, P, I, L, P, I, F, F, F, P, P, P]
        assert fn(gated.data_ptr(), x.data_ptr(), up.data_ptr(), M, width, W, W, width, p.order.data_ptr(), E, 2 * width * W, p.token.data_ptr(), T, limit, slope, shift,
                  *weighed, stream()) == 0
    assert parts(got.data_ptr(), gated.data_ptr(), down.data_ptr(), M, W, width, width, W, p.order.data_ptr(), E, W * width, None, 0, 0, stream()) == 0
    assert torch.equal(gated[held], act[held]) and torch.equal(got[held], want[held]) and int(held.sum()) == T * top
    assert torch.isnan(got[~held]).all()

    chosen, weights = p.idx.cpu().long().flatten(), p.wts.cpu().flatten()
    y = got[p.pair_row.long()].float().cpu()                                             # of a pair, token * top + choice
    for e in (max(range(E), key=lambda j: p.counts[j]), listed[-1]):
        of = (chosen == e).nonzero().flatten()
        f = (x.cpu()[of // top].float() @ up[e].cpu().float().t()).to(BF16).float()
        if form == "squared":
            a = f.clamp(min=0.0) ** 2
        else:
            f = f * (weights[of, None] if form == "weighed" else 1.0)
            g, u = f[:, :width].clamp(max=limit), f[:, width:].clamp(-limit, limit)
            a = g * torch.sigmoid(slope * g) * (u + shift)
        ref = a.to(BF16).float() @ down[e].cpu().float().t()
        # Half a unit of 16 bits, 2^-9, in the activation's elements and in the result's; and the first product's sums, which where they lie between
        # two elements may be rounded the other way.
        assert float((y[of] - ref).norm() / ref.norm()) < 2 ** -8


@pytest.mark.parametrize("matrices,rows,N,K,gated,takes", [
    (26, 40, 1024, 1024, 0, 1), (25, 40, 1024, 1024, 0, 0), (32, 60, 1024, 1024, 0, 1), (31, 60, 1024, 1024, 0, 0), (40, 150, 1024, 1024, 0, 1), (32, 150, 1024, 1024, 0, 0),
    (57, 150, 1024, 1024, 0, 0), (57, 150, 1024, 2048, 0, 1), (76, 150, 1024, 1024, 0, 1), (32, 60, 512, 1024, 1, 1), (32, 60, 384, 1024, 1, 0),
    (512, 60, 256, 1024, 0, 1), (512, 60, 255, 1024, 0, 0), (512, 60, 128, 1024, 1, 1), (512, 60, 127, 1024, 1, 0), (512, 60, 1024, 512, 0, 0), (512, 60, 1024, 1280, 0, 0)])
def test_where_the_lines_lie(matrices, rows, N, K, gated, takes):
    """On 256 units: 0.4, 0.5 and 0.66 of them in workgroups, a round and a third of them; whole chunks, more than one; columns enough for a workgroup."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    for dtype, want in ((BF16, takes), (torch.float32, 0)):
        fn = kern(dtype).lib.vk_gemm_experts_takes
        fn.argtypes = [I, I, I, L, I, I]
        assert fn(matrices * (rows + 127), N, K, K, matrices, gated) == want


@pytest.mark.parametrize("E,top", [(1, 1), (5, 2), (64, 4), (70, 3)])
def test_order_of_a_plan(E, top):
    """Every expert with rows once, with its first row and its rows; the parts before it; up to 64 experts the taller parts first."""
    k, W = kern(BF16), 64
    for T in (40, 3000):
        p = Plan(k, rand((T, W), BF16, 1).cuda(), rand((E, W), BF16, 2).cuda(), top)
        counts, start, order = p.counts, p.start, p.order
        before, heights, seen = 0, [], []
        for tb, first, rows, e in order.tolist():
            assert tb == before
            if rows:
                assert rows == counts[e] and first == int(start[e])
                parts = -(-rows // PART)
                before += parts
                heights.append(-(-rows // parts))
                seen.append(e)
            else:
                assert len(seen) == sum(n > 0 for n in counts)
        assert sorted(seen) == [e for e, n in enumerate(counts) if n]
        assert E > 64 or heights == sorted(heights, reverse=True)
