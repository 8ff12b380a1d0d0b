"""Prompts whose experts' products go by a plan's order: one prompt against its own tokens in portions so small that they go by tiles of 16 rows, and against the
plain implementation.  The three forms of an expert: gated, gated with weights on what it reads, squared ReLU."""
import ctypes

import numpy as np
import pytest
import torch

import pabavik_models
import pasovik_models
import plain_pabavik
import plain_pasovik
import plain_povatar
import povatar_models
from test_kernels_gpu import kern

pytestmark = pytest.mark.gpu
TOKENS = 560


def model(design, W, F, E, top):
    if design == "pabavik":
        m = pabavik_models
        return m, plain_pabavik, m.config([m.layer("gla", m.gla(1, 4, 4), m.moe(E, top, F, limit=1.0, shared=(64, 1.0)))], width=W, vocab=50)
    if design == "pasovik":
        m = pasovik_models
        return m, plain_pasovik, m.config([m.layer("lightning", m.lightning(1, 4, 4, [0.9]), m.moe(E, top, F, limit=1.0))], width=W, vocab=50)
    m = povatar_models
    return m, plain_povatar, m.config([m.layer(m.left(1, 1, 8, 8, size=4, rot_dims=4), m.right(1, 4, 4, 1, 1, conv=2), m.moe(E, top, F))], width=W, vocab=50)


@pytest.mark.parametrize("design", ["pabavik", "pasovik", "povatar"])
@pytest.mark.parametrize("W,F,E,top,up,down", [(1024, 1024, 32, 2, 1, 1), (1024, 512, 64, 4, 1, 0), (512, 1024, 64, 4, 0, 1)], ids=["both", "up_alone", "down_alone"])
def test_a_prompt_and_its_portions(tmp_path, W, F, E, top, up, down, design):
    from vosti_amd.engine.native import NativeEngine
    lib = kern(torch.bfloat16).lib
    lib.vk_moe_max_tiles.argtypes = [ctypes.c_int] * 4
    lib.vk_gemm_experts_takes.argtypes = [ctypes.c_int] * 3 + [ctypes.c_int64] + [ctypes.c_int] * 2
    rows, gated = lib.vk_moe_max_tiles(TOKENS, top, E, 128) * 128, int(design != "povatar")
    assert TOKENS * top >= 32 * E > TOKENS // 2 * top
    assert (lib.vk_gemm_experts_takes(rows, F, W, W, E, gated), lib.vk_gemm_experts_takes(rows, W, F, F, E, 0)) == (up, down)

    m, plain, cfg = model(design, W, F, E, top)
    w = m.random_weights(cfg, 7)
    eng = NativeEngine(m.write_model(tmp_path / design, cfg, w), dtype="bfloat16", num_pages=2 * TOKENS // 16 + 8, page_size=16, max_num_seqs=4, enable_prefix_cache=False,
                       graphs=False)
    tokens = torch.randint(0, cfg["vocab"], (TOKENS,), generator=torch.Generator().manual_seed(2)).tolist()
    half = TOKENS // 2
    whole = eng.trace_step([(0, tokens, list(range(TOKENS)))])
    parts = np.concatenate([eng.trace_step([(1, tokens[at:at + half], list(range(half)))]) for at in (0, half)])
    root = np.sqrt((whole.astype(np.float64) ** 2).mean())
    assert np.sqrt(((whole - parts).astype(np.float64) ** 2).mean(-1)).max() < 2e-5 * root
    if up and down:
        # The products' rounding to 16 bits.  A token whose second and third expert all but tie may be given the other one: the router's input is rounded to 2^-9 of
        # itself, its logits of deviation 2 move by 0.008 at most between them, and of 32 the second and third lie half a unit apart on the mean: two tokens in a hundred.
        want = plain.forward(cfg, w, tokens).numpy()
        off = np.sqrt(((whole - want) ** 2).mean(-1)) / np.sqrt((want ** 2).mean())
        assert np.quantile(off, 0.95) < 6e-2
