"""Chunks on f32 layers whose pages a launch of its own splits into terms (and whose rows it stores), against the oracle and
against the other way, in which each workgroup splits its pages: edges of pairs of pages, contexts in several segments, rings
whose new rows stay in the caller's memory, padded and unaligned heads, infinities. Contexts within 2e-5 (two f32 sums of
up to 600 products in different orders), rows bit for bit."""
import os

import numpy as np
import pytest

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu


def under(env, call):
    env = dict(env, SKV_PREFILL_TILES="2")  # the chunk kernel for every chunk of 64 slots and more
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    skv.flags.reload()
    try:
        return call()
    finally:
        for k, v in saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
        skv.flags.reload()


MADE = {"halves": {"SKV_F32_TERMS": "2"}, "one_tile": {"SKV_F32_TERMS": "2", "SKV_PREFILL_TILES2_MIN_PAGES": "1000000"},
        "segments": {"SKV_F32_TERMS": "2", "SKV_F32_TERMS_MB": "1"}, "no_split": {"SKV_F32_TERMS": "2", "SKV_PREFILL_MAX_SPLITS": "1"},
        "own": {"SKV_F32_TERMS": "0"},
        # chosen, and then no memory for them: the call stores its rows and splits its pages another way
        "refused": {"SKV_F32_TERMS": "2", "SKV_F32_TERMS_MB": "0"}}


@pytest.mark.parametrize("mode", MADE)
@pytest.mark.parametrize("dims,window,base,chunks", [
    ((8, 2, 64), 0, 0, (17, 130)),      # from an empty cache; the last pair has one page
    ((8, 2, 64), 0, 31, (33, 64)),      # base at the end of a page pair
    ((32, 8, 128), 0, 509, (66,)),      # a page shared by cached and new rows; 1 MiB holds two pairs
    ((16, 2, 256), 0, 255, (41, 8)),
    ((6, 1, 40), 0, 1, (11, 43)),       # heads per group not a power of two, padded head
    ((16, 2, 18), 0, 70, (64,)),        # no 16-byte rows
    ((12, 4, 90), 0, 100, (30, 100)),   # padded head whose rows are 8-byte aligned
    ((8, 2, 64), 40, 0, (100, 200)),    # ring: chunk longer than the ring from the start
    ((8, 2, 64), 48, 47, (90, 17)),     # ring: an odd number of old pages, chunk starts inside a page
    ((16, 8, 256), 33, 300, (130,)),
    ((4, 2, 18), 17, 64, (64, 33)),     # ring: chunk starts at a page boundary; padded, unaligned head
])
def test_chunks_of_made_terms(state, mode, dims, window, base, chunks):
    q_heads, kv_heads, head_dim = dims
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(base + head_dim)
    kv = state.full_attention_f32(base + sum(chunks), q_heads, kv_heads, head_dim, window=window)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32")
    if base:
        k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
        kv.seed(k0, v0, base)
        cache.append_batch(k0, v0, lay)
    for c in chunks:
        q = rng.standard_normal((c, q_dim), dtype=np.float32)
        k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
        got = under(MADE[mode], lambda: kv.prefill_rows(q, k, v))
        want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
        assert np.abs(got - want).max() <= 2e-5, c
    first = max(0, kv.len() - window) if window else 0
    gk, gv = kv.read_rows_f32(first, kv.len() - first)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])


@pytest.mark.parametrize("mode", ["halves", "segments", "refused"])
@pytest.mark.parametrize("head_dim,window,base", [(64, 0, 61), (128, 0, 900), (256, 0, 333), (64, 70, 61), (128, 900, 1200)])
def test_infinities_as_in_the_other_way(state, mode, head_dim, window, base):
    """Rows with infinities, and rows that were rolled back and hold NaN: the same contexts either way, and no NaN from rows that
    nobody attends."""
    q_heads, kv_heads, rows = 4, 2, 150
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(head_dim + window)
    k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
    bad = np.full((9, kv_dim), np.nan, dtype=np.float32)
    q = rng.standard_normal((rows, q_dim), dtype=np.float32)
    k, v = (rng.standard_normal((rows, kv_dim), dtype=np.float32) for _ in range(2))
    v[20, 3], v[100, head_dim + 7], v[60, 5] = np.inf, -np.inf, np.float32(3.4e38)
    k[40, 9], k[120, head_dim + 2], q[140, 2 * head_dim + 1] = np.inf, -np.inf, np.inf

    def run():
        kv = state.full_attention_f32(base + rows + 20, q_heads, kv_heads, head_dim, window=window)
        kv.seed(k0, v0, base)
        kv.append_batch(bad, bad) if hasattr(kv, "append_batch") else [kv.append_row(b, b) for b in bad]
        kv.truncate(base)
        return kv.prefill_rows(q, k, v)

    got, want = under(MADE[mode], run), under(MADE["own"], run)
    assert np.isfinite(want[:20]).all() and not np.isfinite(want).all()
    for test in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(test(got), test(want))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= 2e-5 * np.maximum(np.abs(want[ok]), 1.0)).all()


@pytest.mark.parametrize("mode", ["halves", "one_tile", "segments", "no_split", "refused"])
@pytest.mark.parametrize("over", ["k", "v"])
def test_context_over_the_rows_that_the_terms_launch_stores(state, mode, over):
    """The context may lie where the chunk's K or V rows are (a caller's activations share a buffer)."""
    torch = pytest.importorskip("torch")
    q_heads, kv_heads, head_dim, base, rows = 8, 2, 64, 300, 200
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(rows)
    k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
    q, k, v = (rng.standard_normal((rows, d), dtype=np.float32) for d in (q_dim, kv_dim, kv_dim))
    kv = state.full_attention_f32(base + rows, q_heads, kv_heads, head_dim)
    kv.seed(k0, v0, base)
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache = oracle.LayerKvCache("f32")
    cache.append_batch(k0, v0, lay)
    want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
    arena = torch.zeros(rows * q_dim, device="cuda")  # the context's; the rows lie in its end
    shared = torch.from_numpy(k if over == "k" else v).cuda().flatten()
    apart, qd = torch.from_numpy(v if over == "k" else k).cuda(), torch.from_numpy(q).cuda()
    arena[-rows * kv_dim:] = shared
    at = arena.data_ptr() + rows * (q_dim - kv_dim) * 4
    stream = torch.cuda.current_stream().cuda_stream
    under(MADE[mode], lambda: kv.encode_prefill_rows(stream, qd.data_ptr(), at if over == "k" else apart.data_ptr(),
                                                     at if over == "v" else apart.data_ptr(), rows, arena.data_ptr()))
    torch.cuda.synchronize()
    assert np.abs(arena.cpu().numpy().reshape(rows, q_dim) - want).max() <= 2e-5
    gk, gv = kv.read_rows_f32(0, kv.len())
    assert np.array_equal(gk, cache.keys()) and np.array_equal(gv, cache.values())


def test_chunks_of_made_terms_on_two_streams_in_turn(state):
    """Two sequences of one context on streams of their own, whose chunks are in flight together: each has its terms to itself."""
    torch = pytest.importorskip("torch")
    q_heads, kv_heads, head_dim, steps = 16, 4, 64, 5
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    work = []
    for i, rows in enumerate((130, 96)):
        gen = np.random.default_rng(i)
        q, k, v = (gen.standard_normal((steps, rows, d), dtype=np.float32) for d in (q_dim, kv_dim, kv_dim))
        work.append((state.full_attention_f32(steps * rows, q_heads, kv_heads, head_dim), torch.cuda.Stream(), rows, (q, k, v),
                     [torch.from_numpy(x).cuda() for x in (q, k, v)], torch.empty(steps, rows, q_dim, device="cuda")))
    torch.cuda.synchronize()

    def run():
        for step in range(steps):
            for kv, stream, rows, _, (q, k, v), out in work:
                kv.encode_prefill_rows(stream.cuda_stream, q[step].data_ptr(), k[step].data_ptr(), v[step].data_ptr(), rows, out[step].data_ptr())

    under(MADE["halves"], run)
    torch.cuda.synchronize()
    for kv, _, rows, (q, k, v), _, out in work:
        cache = oracle.LayerKvCache("f32")
        for step in range(steps):
            want = oracle.cached_attention_prefill_rows(q[step], k[step], v[step], cache, lay)
            assert np.abs(out[step].cpu().numpy() - want).max() <= 2e-5, step
        gk, gv = kv.read_rows_f32(0, kv.len())
        assert np.array_equal(gk, cache.keys()) and np.array_equal(gv, cache.values())
