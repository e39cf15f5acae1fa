"""Ring layers whose rows still fit the ring, so that no position has taken another's slot: windows that hide the oldest rows, chunks of one
row up to many in each kernel and shape, rollbacks, and the first chunk that wraps. Contexts within 1e-4 of the oracle on bf16 layers
(queries and probabilities carry 16 bits: about 1e-5 of values of order one), within 2e-5 on f32 ones (two f32 sums of up to 300
products in different orders), rows bit for bit."""
import os

import numpy as np
import pytest

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu

WAYS = {"default": {}, "streams": {"SKV_PREFILL_TILES": "0"}, "tiles": {"SKV_PREFILL_TILES": "2"},
        "made": {"SKV_PREFILL_TILES": "2", "SKV_F32_TERMS": "2"}, "two_tiles": {"SKV_PREFILL_TILES": "2", "SKV_PREFILL_TILES2_MIN_PAGES": "0"}}


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("dims,window,slack,base,chunks", [
    ((8, 2, 64), 20, 300, 0, (1, 33, 70, 1, 100, 80, 1, 40)), # 320 rows; the last chunk wraps
    ((8, 2, 64), 170, 150, 95, (66, 6, 150, 90)),             # 320 rows, the window about half of them
    ((12, 4, 96), 40, 200, 37, (80, 64, 30, 100)),
    ((16, 8, 256), 64, 200, 1, (130, 70, 90)),                # 272 rows
    ((4, 2, 320), 33, 200, 40, (64, 1, 100, 60)),             # heads above 256
    ((4, 2, 18), 17, 250, 20, (64, 33, 100, 90)),             # no 16-byte rows
])
@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
def test_chunks_before_the_ring_wraps(state, way, element, tol, dims, window, slack, base, chunks):
    q_heads, kv_heads, head_dim = dims
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(base + head_dim)
    kv = state.full_attention_with_element(base + sum(chunks) + 9, q_heads, kv_heads, head_dim,
                                           skv.DTYPE_F32 if element == "f32" else skv.DTYPE_BF16, window, rollback_rows=slack)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    if base:
        k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
        kv.seed(k0, v0, base)
        cache.append_batch(k0, v0, lay)
    saved = {k: os.environ.get(k) for k in WAYS[way]}
    os.environ.update(WAYS[way])
    skv.flags.reload()
    try:
        for c in chunks:
            q = rng.standard_normal((c, q_dim), dtype=np.float32)
            k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
            got = kv.prefill_rows(q, k, v)
            want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
            assert np.abs(got - want).max() <= tol, c
            # rows that are rolled back again and hold NaN must not be seen behind it
            n = kv.len()
            bad = np.full(kv_dim, np.nan, dtype=np.float32)
            if n + 3 <= slack:
                for _ in range(3):
                    kv.append_row(bad, bad)
                kv.truncate(n)
    finally:
        for k, v in saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
        skv.flags.reload()
    first = max(0, kv.len() - window)
    gk, gv = kv.read_rows_f32(first, kv.len() - first)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])
