"""Heads of 65 to 96 dims, whose tiles hold 96: decode steps, few rows and chunks in each workgroup shape, at both ends of the
range and with rows that 16-byte loads cannot read. Contexts within 1e-4 of the oracle on bf16 layers (queries and probabilities carry 16
bits: about 1e-5 of values of order one), within 2e-5 on f32 ones (two f32 sums of up to 400 products in different orders), rows bit for bit;
and the bytes of a layer, which callers budget by, stay those of 128 dims."""
import os

import numpy as np
import pytest

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu

SHAPES = {"default": {}, "one_tile": {"SKV_PREFILL_TILES": "2", "SKV_PREFILL_TILES2_MIN_PAGES": "1000000", "SKV_F32_TERMS": "0"},
          "two_tiles": {"SKV_PREFILL_TILES": "2", "SKV_PREFILL_TILES2_MIN_PAGES": "0", "SKV_F32_TERMS": "2"},
          "halves": {"SKV_PREFILL_TILES": "2", "SKV_F32_TERMS": "2"}, "own": {"SKV_PREFILL_TILES": "2", "SKV_F32_TERMS": "0"}}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dims,window,base", [((6, 2, 65), 0, 37), ((10, 2, 88), 0, 205), ((12, 4, 96), 0, 144), ((12, 4, 96), 50, 77),
                                              ((3, 1, 70), 33, 8)])
@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
def test_rows_and_contexts(state, shape, element, tol, dims, window, base):
    q_heads, kv_heads, head_dim = dims
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    chunks = (1, 7, 66, 1, 130)
    rng = np.random.default_rng(base + head_dim)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(base + sum(chunks), q_heads, kv_heads, head_dim, window=window)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
    kv.seed(k0, v0, base)
    cache.append_batch(k0, v0, lay)
    saved = {k: os.environ.get(k) for k in SHAPES[shape]}
    os.environ.update(SHAPES[shape])
    skv.flags.reload()
    try:
        for c in chunks:
            q = rng.standard_normal((c, q_dim), dtype=np.float32)
            k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
            got = kv.prefill_rows(q, k, v)
            want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
            assert np.abs(got - want).max() <= tol, c
    finally:
        for k, v in saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
        skv.flags.reload()
    first = max(0, kv.len() - window) if window else 0
    gk, gv = kv.read_rows_f32(first, kv.len() - first)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])


def test_layer_bytes():
    for dtype in (skv.DTYPE_BF16, skv.DTYPE_F32):
        a, b = (skv.flags.layer_bytes(4096, 8, 8, hd, dtype) for hd in (96, 128))
        assert 0 <= b - a < 1 << 20  # (the partials and the staged rows are of head_dim itself)
