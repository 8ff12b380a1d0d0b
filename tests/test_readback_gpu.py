"""Logits on their way to the host: one piece and many, whole vectors and not."""
import ctypes

import numpy as np
import pytest
import torch
from test_kernels_gpu import DTYPES, kern, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,shift", [(1, 0), (8, 0), (255, 0), (4096, 0), (4096, 1), (70001, 3), (600000, 0)])
def test_elements_arrive_whole(n, shift, dtype):
    k = kern(dtype)
    x = rand((n + shift,), dtype, 1).cuda()
    out = torch.full((n + shift + 1,), 7.0, dtype=dtype).pin_memory()
    k.lib.vk_copy_out.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]
    at = shift * x.element_size()
    assert k.lib.vk_copy_out(out.data_ptr() + at, x.data_ptr() + at, n, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out[shift:-1], x[shift:].cpu()) and bool((out[:shift] == 7.0).all()) and out[-1] == 7.0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rows_beyond_the_pinned_places(tmp_path, dtype):
    """More rows than the places hold at once (2.5 million and 5 million elements), against the same rows a few at a time."""
    from vosti_amd.config import Qwen3Config
    from vosti_amd.engine import create_engine
    from vosti_amd.weights import write_random_model
    tokens = 4500 if dtype == "float32" else 9100
    cfg = Qwen3Config(vocab_size=555, hidden_size=64, intermediate_size=64, num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=1,
                      head_dim=32, max_position_embeddings=16384, rms_norm_eps=1e-5, rope_theta=1e6, tie_word_embeddings=False)
    write_random_model(cfg, 1, tmp_path)
    engine = create_engine(str(tmp_path), dtype=dtype, num_pages=300, page_size=64, max_num_seqs=2, max_num_batched_tokens=16384)
    ids = np.random.default_rng(1).integers(0, 555, tokens).tolist()
    whole = engine.trace_step([(1, ids, list(range(tokens)))])
    some = [0, 1, 2, 1000, 1889, 1890, 3777, 3778, 4444, tokens - 2, tokens - 1]
    few = engine.trace_step([(2, ids, some)])
    assert whole.shape == (tokens, 555) and np.array_equal(whole[some], few)
    assert np.isfinite(whole).all() and len(np.unique(whole[:, 0])) > 100
