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


def wrapped_and_back(state, element, dims, window, slack, n, seed):
    """A ring that wrapped over its oldest slots with rows of NaN and was rolled back to n rows, few enough to lie in slots of
    their own again (floor_pos > 0); its oracle; its generator."""
    q_heads, kv_heads, head_dim = dims
    kv_dim = kv_heads * head_dim
    rng = np.random.default_rng(seed)
    dtype = skv.DTYPE_F32 if element == "f32" else skv.DTYPE_BF16
    kv = state.full_attention_with_element(4 * (window + slack), q_heads, kv_heads, head_dim, dtype, window, rollback_rows=slack)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    ring = kv.pages() * 16
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    k0, v0 = (rng.standard_normal((n, kv_dim), dtype=np.float32) for _ in range(2))
    kv.seed(k0, v0, n)
    cache.append_batch(k0, v0, lay)
    bad = np.full(kv_dim, np.nan, dtype=np.float32)
    while kv.len() < ring + n + 1 - window:  # the last one takes the slot in front of the oldest row that the next query attends
        kv.append_row(bad, bad)
    assert n <= ring < kv.len()
    kv.truncate(n)
    return kv, cache, lay, rng, ring


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("dims,window,slack,n", [((8, 2, 64), 230, 10, 236), ((12, 4, 96), 150, 42, 170), ((16, 8, 256), 100, 44, 130),
                                                 ((4, 2, 320), 70, 26, 90)])
@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
def test_rings_rolled_back_to_before_they_wrapped(state, way, element, tol, dims, window, slack, n):
    kv, cache, lay, rng, ring = wrapped_and_back(state, element, dims, window, slack, n, n + dims[2])
    q_dim, kv_dim = dims[0] * dims[2], dims[1] * dims[2]
    saved = {k: os.environ.get(k) for k in WAYS[way]}
    os.environ.update(WAYS[way])
    skv.flags.reload()
    try:
        for c in (1, ring - n - 1, 70, 3, 1):  # a row, as many as the ring holds without wrapping, a chunk that wraps, few rows, a row
            q = rng.standard_normal((c, q_dim), dtype=np.float32)
            k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
            got = kv.prefill_rows(q, k, v)
            want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
            assert np.abs(got - want).max() <= tol, c
    finally:
        for k, v in saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
        skv.flags.reload()
    first = kv.len() - window
    gk, gv = kv.read_rows_f32(first, window)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])


@pytest.mark.parametrize("dims", [(8, 2, 64), (16, 8, 256)])
@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
def test_batch_of_rings_in_every_state(state, element, tol, dims):
    """One launch over a ring that was rolled back to before it wrapped, a fresh one and one that has wrapped."""
    torch = pytest.importorskip("torch")
    window, slack, n = 100, 44, 130
    q_dim, kv_dim = dims[0] * dims[2], dims[1] * dims[2]
    kv, cache, lay, rng, ring = wrapped_and_back(state, element, dims, window, slack, n, 7)
    seqs = [(kv, cache, lay)]
    for rows in (20, 400):
        dtype = skv.DTYPE_F32 if element == "f32" else skv.DTYPE_BF16
        other = state.full_attention_with_element(500, *dims, dtype, window, rollback_rows=slack)
        cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
        k0, v0 = (rng.standard_normal((rows, kv_dim), dtype=np.float32) for _ in range(2))
        other.seed(k0, v0, rows)
        cache.append_batch(k0, v0, lay)
        seqs.append((other, cache, lay))
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(ring - n + 2):  # until the first one wraps again
        rows = [[rng.standard_normal(d, dtype=np.float32) for d in (kv_dim, kv_dim, q_dim)] for _ in seqs]
        dev = [[torch.from_numpy(a).cuda() for a in r] for r in rows]
        outs = [torch.empty(q_dim, device="cuda") for _ in seqs]
        skv.encode_decode_step_batch([s[0] for s in seqs], stream, *([d[i].data_ptr() for d in dev] for i in range(3)),
                                     [o.data_ptr() for o in outs])
        for (_, cache, lay), (k, v, q), o in zip(seqs, rows, outs):
            assert np.abs(o.cpu().numpy() - oracle.decode_step(cache, k, v, q, lay)).max() <= tol
