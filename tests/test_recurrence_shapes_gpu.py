"""The recurrences' kernels for whole vectors (prompts in chunks, steps of single tokens) against the walk that takes every shape, which
rows of an odd length lead to: the same bits in the read-outs and the states, whatever the lengths; and both against the equations."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern

pytestmark = pytest.mark.gpu


def unit_heads(x, kind, G, d):
    """The delta rule's q and k as it meets them, of unit length a head; with others its corrections grow from token to token."""
    if kind == "delta":
        heads = x[:, :2 * G * d].view(x.shape[0], 2 * G, d)
        heads /= heads.norm(dim=-1, keepdim=True)


def run(k, kind, d, heads, lengths, fresh, odd, dtype):
    """One step of sequences of these lengths; odd: rows one element longer, so that they are not whole vectors."""
    g = torch.Generator().manual_seed(3)
    T, S, H, dv = sum(lengths), len(lengths), heads, 128
    G = H // 2 if kind == "delta" else H
    cols = 2 * G * d + H * dv
    x = torch.randn(T, cols, generator=g)
    unit_heads(x, kind, G, d)
    rows = torch.zeros(T, cols + (1 if odd else 0))
    rows[:, :cols] = x
    rows = rows.to(torch.float32 if kind == "delta" else dtype).cuda()
    decay = (0.9 + 0.1 * torch.rand(T, H, d, generator=g)).cuda()
    head_decay = (0.9 + 0.1 * torch.rand(H, generator=g)).cuda()
    beta = torch.randn(T, H, generator=g).to(dtype).cuda()
    state = torch.randn(S + 1, H * d * dv, generator=g).cuda()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    positions = torch.arange(T, dtype=torch.int32) + (0 if fresh else 7)
    for s in range(S):
        positions[cu[s]] = 0 if fresh and s % 2 == 0 else 5
    cu, positions, slots = i32(cu), positions.cuda(), i32([(s + 1) % (S + 1) for s in range(S)])
    out = torch.full((T, H, dv), float("nan"), device="cuda")
    p, i, l, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
    stream = torch.cuda.current_stream().cuda_stream
    where = (cu.data_ptr(), positions.data_ptr(), slots.data_ptr(), T, S, H)
    if kind == "delta":
        fn = k.lib.vk_delta_rule
        fn.argtypes = [p, p, l, i, i, i, p, p, l, p, l, p, p, p, i, i, i, i, i, i, p]
        rc = fn(out.data_ptr(), rows.data_ptr(), rows.shape[1], 0, G * d, 2 * G * d, decay.data_ptr(), beta.data_ptr(), H, state.data_ptr(), state.shape[1],
                *where, G, d, dv, stream)
    else:
        fn = k.lib.vk_gla_rule if kind == "gla" else k.lib.vk_linear_rule
        fn.argtypes = [p, p, l, i, i, i, p, p, l, p, p, p, i, i, i, i, i, f, p]
        rc = fn(out.data_ptr(), rows.data_ptr(), rows.shape[1], 0, H * d, 2 * H * d, (decay if kind == "gla" else head_decay).data_ptr(), state.data_ptr(),
                state.shape[1], *where, d, dv, 0.3, stream)
    assert rc == 0
    torch.cuda.synchronize()
    return out.cpu(), state.cpu()


def plain(kind, d, heads, n, dtype):
    """The read-outs of one sequence from a zero state, for run()'s numbers, in 64 bits."""
    g = torch.Generator().manual_seed(3)
    H, dv = heads, 128
    G = H // 2 if kind == "delta" else H
    x = torch.randn(n, 2 * G * d + H * dv, generator=g)
    unit_heads(x, kind, G, d)
    x = x.to(torch.float32 if kind == "delta" else dtype).double()
    decay = (0.9 + 0.1 * torch.rand(n, H, d, generator=g)).double()
    head_decay = (0.9 + 0.1 * torch.rand(H, generator=g)).double()
    beta = torch.randn(n, H, generator=g).to(dtype).double().sigmoid()
    if kind == "linear":
        decay = head_decay[None, :, None].expand(n, H, d)
    q, key = (x[:, j * G * d:(j + 1) * G * d].view(n, G, d).repeat_interleave(H // G, 1) for j in (0, 1))
    v = x[:, 2 * G * d:].view(n, H, dv)
    S, out = torch.zeros(H, d, dv).double(), []
    for t in range(n):
        S = decay[t][:, :, None] * S
        u = beta[t][:, None] * (v[t] - (S * key[t][:, :, None]).sum(1)) if kind == "delta" else v[t]
        S = S + key[t][:, :, None] * u[:, None, :]
        out.append((S * q[t][:, :, None]).sum(1) * (1.0 if kind == "delta" else 0.3))
    return torch.stack(out)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [8, 16, 40, 64, 100, 128, 200, 300])
@pytest.mark.parametrize("kind", ["delta", "gla", "linear"])
def test_the_equations(kind, d, dtype):
    """Sums over 1 to 64 lanes.  Everything is 32-bit: 45 tokens of a decayed sum of products are good to a few 1e-7 of their size."""
    got, want = run(kern(dtype), kind, d, 2, [45], True, False, dtype)[0].double(), plain(kind, d, 2, 45, dtype)
    assert (got - want).norm() < 5e-6 * want.norm()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["delta", "gla", "linear"])
def test_the_same_bits_as_the_walk_for_every_shape(kind, d, dtype):
    k = kern(dtype)
    for heads, lengths, fresh in ((4, [1], True), (4, [1, 1, 1], True), (4, [1, 1, 1], False), (4, [16], True), (4, [15, 1, 17], False), (4, [33, 2, 48], True),
                                  (48, [17, 5, 32], False)):           # the last: so many workgroups that a lane takes two columns
        got, want = (run(k, kind, d, heads, lengths, fresh, odd, dtype) for odd in (False, True))
        assert not torch.isnan(got[0]).any()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["delta", "gla", "linear"])
def test_uneven_steps_of_as_many_tokens_as_sequences(kind, d, dtype):
    """Not one token each: the bits of the walk for every shape, and the states of sequences without a token as they were."""
    for lengths in ([0, 2], [2, 0, 1], [0, 0, 3], [0, 1, 3, 0, 1]):
        got, want = (run(kern(dtype), kind, d, 4, lengths, False, odd, dtype) for odd in (False, True))
        assert not torch.isnan(got[0]).any()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def run_scan(k, heads, P, lengths, fresh, odd):
    """The state-space scan with 128 state rows over sequences of these lengths; odd: rows one number longer."""
    g = torch.Generator().manual_seed(4)
    T, S, H, N, G = sum(lengths), len(lengths), heads, 128, 2
    cols = H * P + 2 * G * N
    rows = torch.zeros(T, cols + (1 if odd else 0))
    rows[:, :cols] = torch.randn(T, cols, generator=g)
    dt = torch.randn(T, H, generator=g).to(k.dtype)
    bias, A_log, D = (torch.rand(H, generator=g) for _ in range(3))
    state = torch.randn(S + 1, H * P * N, generator=g)
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    positions = torch.arange(T, dtype=torch.int32)
    for s in range(S):
        positions[cu[s]] = 0 if fresh and s % 2 == 0 else 5
    slots = [(s + 1) % (S + 1) for s in range(S)]
    want = None
    if lengths == [45]:
        z = dt.double() + bias.double()
        step = torch.nn.functional.softplus(z)
        decay = torch.exp(-torch.exp(A_log.double()) * step)
        St, want = torch.zeros(H, N, P).double(), []
        for t in range(T):
            row = rows[t].double()
            x, B, C = row[:H * P].view(H, P), row[H * P:H * P + G * N].view(G, N), row[H * P + G * N:H * P + 2 * G * N].view(G, N)
            B, C = B.repeat_interleave(H // G, 0), C.repeat_interleave(H // G, 0)
            St = decay[t][:, None, None] * St + step[t][:, None, None] * B[:, :, None] * x[:, None, :]
            want.append((St * C[:, :, None]).sum(1) + D.double()[:, None] * x)
        want = torch.stack(want)
    dev = [v.cuda() for v in (rows, dt, bias, A_log, D, state, torch.tensor(cu, dtype=torch.int32), positions, torch.tensor(slots, dtype=torch.int32))]
    rows, dt, bias, A_log, D, state, cu, positions, slots = dev
    y = torch.full((T, H, P), float("nan"), device="cuda")
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_ssm_scan
    fn.argtypes = [p, p, l, i, i, p, l, p, p, p, i, p, l, p, p, p, i, i, i, i, i, i, p]
    assert fn(y.data_ptr(), rows.data_ptr(), rows.shape[1], H * P, H * P + G * N, dt.data_ptr(), H, bias.data_ptr(), A_log.data_ptr(), D.data_ptr(), 1,
              state.data_ptr(), state.shape[1], cu.data_ptr(), positions.data_ptr(), slots.data_ptr(), S, T, H, G, N, P,
              torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return y.cpu(), state.cpu(), want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("P", [48, 64])
def test_the_state_space_scan(P, dtype):
    k = kern(dtype)
    for heads, lengths, fresh in ((2, [45], True), (2, [1], True), (4, [1, 1, 1], False), (4, [16], True), (4, [15, 1, 17], False), (4, [33, 2, 48], True),
                                  (64, [17, 5, 32], False)):           # the last: so many workgroups that a lane takes two columns
        (y, state, want), (y2, state2, _) = run_scan(k, heads, P, lengths, fresh, False), run_scan(k, heads, P, lengths, fresh, True)
        assert not torch.isnan(y).any()
        assert torch.equal(y, y2) and torch.equal(state, state2)
        if want is not None:                               # 32-bit sums of 128 products and 45 decayed terms
            assert (y.double() - want).norm() < 5e-6 * want.norm()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K,C,with_bias", [(2, 1028, False), (3, 64, True), (4, 260, False), (4, 96, True), (6, 96, False), (1, 40, False)])
def test_the_short_convolution(K, C, with_bias, dtype):
    """Groups of 16 tokens within a sequence, across sequences and at the end; single tokens with their tails; against the sums written out
    with the tails that the step before left."""
    k = kern(dtype)
    g = torch.Generator().manual_seed(5)
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    taps = (0.4 * torch.randn(C, K, generator=g)).to(dtype)
    bias = (0.2 * torch.randn(C, generator=g)).to(dtype)
    fn = k.lib.vk_delta_conv_bias if with_bias else k.lib.vk_delta_conv
    fn.argtypes = [p, p, l, p] + ([p] if with_bias else []) + [p, l, l, p, p, p, p, i, i, i, i, p]
    offset, S = 8, 4
    state = torch.randn(S, offset + 32 + max(K - 1, 1) * C, generator=g).cuda()
    fed = [[] for _ in range(S)]
    for lengths in ([40, 1, 17, 2], [1, 1, 1, 1], [16, 3, 33, 1], [1, 1, 1, 1]):
        T = sum(lengths)
        x = torch.randn(T, C + 8, generator=g).to(dtype)
        cu = [0]
        for n in lengths:
            cu.append(cu[-1] + n)
        positions, seq, want = torch.zeros(T, dtype=torch.int32), torch.zeros(T, dtype=torch.int32), []
        for s in range(S):
            positions[cu[s]:cu[s + 1]] = torch.arange(lengths[s], dtype=torch.int32) + len(fed[s])
            seq[cu[s]:cu[s + 1]] = s
            for t in range(cu[s], cu[s + 1]):
                fed[s].append(x[t, :C].double())
                z = (bias.double() if with_bias else torch.zeros(C).double()) + sum(
                    taps[:, j].double() * fed[s][len(fed[s]) - K + j] for j in range(K) if len(fed[s]) - K + j >= 0)
                want.append(z * torch.sigmoid(z))
        y = torch.full((T, C), float("nan"), device="cuda")
        xs, tg, bg = x.cuda(), taps.cuda(), bias.cuda()
        i32 = [v.to(torch.int32).cuda() for v in (seq, torch.tensor(cu), positions, torch.arange(S))]
        args = (y.data_ptr(), xs.data_ptr(), xs.shape[1], tg.data_ptr()) + ((bg.data_ptr(),) if with_bias else ())
        assert fn(*args, state.data_ptr(), state.shape[1], offset, *(v.data_ptr() for v in i32), T, S, C, K, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        # 32-bit sums of up to six products and a logistic function.
        assert (y.cpu().double() - torch.stack(want)).abs().max() < 2e-5


def test_more_channels_than_a_grid_of_groups():
    """More than 65,535 groups of 256 channels: as many sequences as tokens, and fewer, against the same channels in two halves."""
    k, K = kern(torch.bfloat16), 2
    C = 256 * 65535 + 512
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_delta_conv
    fn.argtypes = [p, p, l, p, p, l, l, p, p, p, p, i, i, i, i, p]
    g = torch.Generator(device="cuda").manual_seed(7)
    for T in (1, 3):
        x, taps = (torch.randn(n, C, device="cuda", generator=g).to(torch.bfloat16) for n in (T, K))
        taps = taps.T.contiguous()
        seq, cu, positions, slots = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([0] * T, [0, T], [1 + t for t in range(T)], [0]))
        tail = torch.randn(1, C, device="cuda", generator=g)
        outs = []
        for cuts in ((0, C), (0, C // 2, C)):
            state, y = tail.clone(), torch.full((T, C), float("nan"), device="cuda")
            for a, b in zip(cuts, cuts[1:]):
                part, tails = (y if b - a == C else y[:, a:b].contiguous()), state[:, a:b].contiguous()
                assert fn(part.data_ptr(), x[:, a:].data_ptr(), C, taps[a:b].contiguous().data_ptr(), tails.data_ptr(), b - a, 0, seq.data_ptr(), cu.data_ptr(),
                          positions.data_ptr(), slots.data_ptr(), T, 1, b - a, K, torch.cuda.current_stream().cuda_stream) == 0
                y[:, a:b], state[:, a:b] = part, tails
            outs.append((y, state))
        assert not torch.isnan(outs[0][0]).any()
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K,with_bias", [(2, False), (3, True), (4, False), (4, True)])
def test_many_channels_at_once_and_few(K, with_bias, dtype):
    """Tokens times channels choose the kernel: all channels in one call and in pieces of 1,028 give the same bits and tails, for groups of 16 tokens within
    a sequence, across several and at the end."""
    k, C, piece, offset = kern(dtype), 32896, 1028, 8
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_delta_conv_bias if with_bias else k.lib.vk_delta_conv
    fn.argtypes = [p, p, l, p] + ([p] if with_bias else []) + [p, l, l, p, p, p, p, i, i, i, i, p]
    g = torch.Generator(device="cuda").manual_seed(9)
    new = lambda *n: torch.randn(*n, device="cuda", generator=g)
    taps, bias = (0.4 * new(C, K)).to(dtype), (0.2 * new(C)).to(dtype)
    for lengths in ([64], [40, 1, 17, 6], [1] * 9 + [2, 33, 21]):
        T, S = sum(lengths), len(lengths)
        assert T * C >= 1 << 21 > T * piece
        x = new(T, C).to(dtype)
        cu = [0]
        for n in lengths:
            cu.append(cu[-1] + n)
        positions = [(0 if s % 2 else 3) + t for s, n in enumerate(lengths) for t in range(n)]
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
        where = [i32(v) for v in ([s for s, n in enumerate(lengths) for _ in range(n)], cu, positions, list(range(S))[::-1])]
        tails = new(S, K - 1, C)
        outs = []
        for step in (C, piece):
            y, after = torch.full((T, C), float("nan"), device="cuda"), torch.zeros_like(tails)
            for a in range(0, C, step):
                n = min(step, C - a)
                part, here = torch.full((T, n), float("nan"), device="cuda"), x[:, a:a + n].contiguous()
                state = torch.zeros(S, offset + (K - 1) * n, device="cuda")
                state[:, offset:] = tails[:, :, a:a + n].reshape(S, -1)
                tp, bs = taps[a:a + n].contiguous(), bias[a:a + n].contiguous()
                args = (part.data_ptr(), here.data_ptr(), n, tp.data_ptr()) + ((bs.data_ptr(),) if with_bias else ())
                assert fn(*args, state.data_ptr(), state.shape[1], offset, *(v.data_ptr() for v in where), T, S, n, K,
                          torch.cuda.current_stream().cuda_stream) == 0
                y[:, a:a + n], after[:, :, a:a + n] = part, state[:, offset:].view(S, K - 1, n)
            outs.append((y, after))
        assert not torch.isnan(outs[0][0]).any()
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("K", [2, 4, 6])
@pytest.mark.parametrize("lengths", [[0, 2], [2, 0, 1], [0, 0, 3], [1, 4, 0, 0, 0]])
def test_the_short_convolution_of_uneven_steps(lengths, K, dtype):
    """As many tokens as sequences, but not one each: the bits and tails of a call a sequence; a sequence without tokens keeps its tail."""
    k, C = kern(dtype), 300
    p, i, l = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    fn = k.lib.vk_delta_conv
    fn.argtypes = [p, p, l, p, p, l, l, p, p, p, p, i, i, i, i, p]
    g = torch.Generator().manual_seed(11)
    S = len(lengths)
    T = sum(lengths)
    x, taps = torch.randn(T, C, generator=g).to(dtype).cuda(), (0.4 * torch.randn(C, K, generator=g)).to(dtype).cuda()
    tails = torch.randn(S, (K - 1) * C, generator=g).cuda()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")

    def step(a, counts, slots, state):
        """The tokens from a on, as sequences of these lengths in these slots; every second slot's sequence starts here."""
        cu, n = [0], sum(counts)
        for c in counts:
            cu.append(cu[-1] + c)
        seq = [s for s, c in enumerate(counts) for _ in range(c)]
        positions = [(5 if slots[s] % 2 else 0) + j for s, c in enumerate(counts) for j in range(c)]
        y, keep = torch.full((n, C), float("nan"), device="cuda"), [x[a:a + n].contiguous(), i32(seq), i32(cu), i32(positions), i32(slots)]
        assert fn(y.data_ptr(), keep[0].data_ptr(), C, taps.data_ptr(), state.data_ptr(), state.shape[1], 0, *(v.data_ptr() for v in keep[1:]), n, len(counts),
                  C, K, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return y

    state, want = tails.clone(), tails.clone()
    y = step(0, lengths, list(range(S)), state)
    at = [sum(lengths[:s]) for s in range(S)]
    rows = torch.cat([step(at[s], [n], [s], want) for s, n in enumerate(lengths) if n])
    assert torch.equal(y, rows) and torch.equal(state, want)
