"""What follows a sublayer in one launch, against the launches that it stands for: the same bits."""
import ctypes

import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu
P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
SIZES = [(1, 4), (3, 1020), (2, 1024), (5, 1028), (1, 2048), (3, 2052), (2, 4096), (1, 4100), (2, 8192)]


def stream():
    return torch.cuda.current_stream().cuda_stream


def call(k, name, types, *args):
    fn = getattr(k.lib, name)
    fn.argtypes = types
    assert fn(*(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args)) == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,H", SIZES)
@pytest.mark.parametrize("y_f32,n", [(False, 0), (True, 0), (False, 1), (False, 2), (True, 9)])
def test_norm_add_mix_and_norm(rows, H, y_f32, n, dtype):
    """A norm added to the stream and the next norm, without and with the weighted sum of 1, 2 and 9 states; weights of both types; the stream in place."""
    k = kern(dtype)
    y = rand((rows, H), torch.float32 if y_f32 else dtype, 1).cuda()
    w, w2 = rand((H,), dtype, 2).cuda(), rand((H,), torch.float32, 3).cuda()
    base, states, coef = rand((rows, H), torch.float32, 4).cuda(), rand((max(n, 1), rows, H), torch.float32, 5).cuda(), rand((max(n, 1),), torch.float32, 6).cuda()
    want_out = torch.empty(rows, H, device="cuda")
    call(k, "vk_stream_norm_add_f32" if y_f32 else "vk_stream_norm_add", [P, P, P, P, I, I, I, F, F, F, P], want_out, base, y, w, w.dtype == torch.float32, rows, H,
         1e-5, 1.0, 0.5, stream())
    want_states, want_mixed = states.clone(), want_out
    if n:
        want_states[n - 1] = want_out
        want_mixed = torch.empty_like(want_out)
        call(k, "vk_stream_mix", [P, P, L, P, I, I, L, P], want_mixed, want_states, rows * H, coef, 1, n, rows * H, stream())
    want = norm(k, want_mixed, w2, 1e-6, 1.0)
    out = states[n - 1] if n else base.clone()
    mixed, normed = torch.empty(rows, H, device="cuda"), torch.empty(rows, H, dtype=dtype, device="cuda")
    call(k, "vk_stream_norm_step", [P, P, P, I, P, I, I, I, F, F, F, P, P, L, P, I, I, P, P, I, F, F, P], out, base if n else out, y, y.dtype == torch.float32, w,
         w.dtype == torch.float32, rows, H, 1e-5, 1.0, 0.5, mixed if n else None, states if n else None, rows * H, coef if n else None, 1, n, normed, w2, 1,
         1e-6, 1.0, stream())
    assert torch.equal(out, want_out) and torch.equal(normed, want) and (not n or torch.equal(mixed, want_mixed))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,H", SIZES)
def test_sum_and_two_norms(rows, H, dtype):
    k = kern(dtype)
    x, a, b = (rand((rows, H), torch.float32, i).cuda() for i in (1, 2, 3))
    w1, w2 = rand((H,), dtype, 4).cuda(), rand((H,), torch.float32, 5).cuda()
    want = x.clone()
    call(k, "vk_stream_add", [P, P, P, I, P, I, L, P], want, want, a, 1, b, 1, rows * H, stream())
    o1, o2 = (torch.empty(rows, H, dtype=dtype, device="cuda") for _ in range(2))
    call(k, "vk_stream_sum_norms", [P, P, P, I, I, P, P, I, F, F, P, P, I, F, F, P], x, a, b, rows, H, o1, w1, w1.dtype == torch.float32, 1e-5, 1.0, o2, w2, 1, 1e-6, 0.0,
         stream())
    assert torch.equal(x, want) and torch.equal(o1, norm(k, want, w1, 1e-5, 1.0)) and torch.equal(o2, norm(k, want, w2, 1e-6, 0.0))


def norm(k, x, w, eps, offset):
    """The norm of the stream's own kernels, whatever the element type."""
    out = torch.empty(x.shape, dtype=k.dtype, device="cuda")
    call(k, "vk_stream_norm", [P, P, I, P, I, I, I, F, F, P], out, x, 1, w, w.dtype == torch.float32, x.shape[0], x.shape[1], eps, offset, stream())
    return out


def test_sizes_that_do_not_fit_are_refused():
    k = kern(torch.bfloat16)
    assert [k.lib.vk_stream_step_takes(h) for h in (0, 4, 6, 8192, 8196)] == [0, 1, 0, 1, 0]
