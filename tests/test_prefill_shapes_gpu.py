"""The prefill kernels of both elements in each of its workgroup shapes, at the edges of its tiles: chunks that end
inside a slot tile, a page pair and a barrier step; caches that begin the chunk inside a page; ring
layers whose chunk starts before, at and long after the ring is full (its rows are attended
from pages of their own and appended afterwards). Contexts within 1e-4 of the oracle on bf16 layers
(queries and probabilities carry 16 bits: about 1e-5 of values of order one), within 2e-5 on f32 ones
(two f32 sums of up to 600 products in different orders), rows bit for bit."""
import os

import numpy as np
import pytest

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu

SHAPES = {"halves": {}, "one_tile": {"SKV_PREFILL_TILES2_MIN_PAGES": "1000000"}, "two_tiles": {"SKV_PREFILL_TILES2_MIN_PAGES": "0"}}


@pytest.fixture(params=SHAPES, ids=str)
def shape(request):
    env = dict(SHAPES[request.param], SKV_PREFILL_TILES="2")  # the tile kernel for every chunk of 64 slots and more
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    skv.flags.reload()
    yield request.param
    for k, v in saved.items():
        os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
    skv.flags.reload()


@pytest.mark.parametrize("dims,window,base,chunks", [
    ((4, 2, 16), 0, 0, (33, 64)),        # the narrowest head, from an empty cache
    ((8, 2, 64), 0, 31, (17, 130)),      # base at the end of a page pair
    ((4, 1, 80), 0, 5, (16, 65)),        # padded head, slots in one tile row and one more
    ((32, 8, 128), 0, 509, (66,)),       # splits of unequal length
    ((16, 2, 256), 0, 255, (41, 8)),
    ((6, 1, 40), 0, 1, (11, 43)),        # heads per group not a power of two, 66 and 258 slots
    ((4, 1, 320), 0, 77, (16, 40)),      # wide heads
    ((8, 2, 64), 40, 0, (100, 200)),     # ring: chunk longer than the ring from the start
    ((8, 2, 64), 48, 47, (90, 17)),      # ring: window of whole pages, chunk starts inside a page
    ((16, 8, 256), 33, 300, (130,)),
    ((4, 2, 16), 17, 64, (64, 33)),      # ring: chunk starts at a page boundary; padded head
])
@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
def test_chunks_in_every_shape(state, shape, element, tol, dims, window, base, chunks):
    q_heads, kv_heads, head_dim = dims
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(base + head_dim)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(base + sum(chunks), q_heads, kv_heads, head_dim, window=window)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    if base:
        k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
        kv.seed(k0, v0, base)
        cache.append_batch(k0, v0, lay)
    for c in chunks:
        q = rng.standard_normal((c, q_dim), dtype=np.float32)
        k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
        got = kv.prefill_rows(q, k, v)
        want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
        assert np.abs(got - want).max() <= tol, (shape, c)
    first = max(0, kv.len() - window) if window else 0
    gk, gv = kv.read_rows_f32(first, kv.len() - first)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])
    kv.close()


@pytest.mark.parametrize("element", ["bf16", "f32"])
def test_scores_that_climb(state, shape, element):
    """Keys that grow along the context move the softmax base again and again (it follows a slot's
    scores only once they pass it), and fall below it by far more."""
    rng = np.random.default_rng(3)
    q_heads, kv_heads, head_dim, n = 8, 2, 64, 300
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(n, q_heads, kv_heads, head_dim)
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    q = np.abs(rng.standard_normal((n, q_heads * head_dim), dtype=np.float32))
    scale = np.linspace(0.0, 9.0, n, dtype=np.float32)[:, None] * np.where(np.arange(n) % 3 == 0, -1.0, 1.0).astype(np.float32)[:, None]
    k = np.abs(rng.standard_normal((n, kv_heads * head_dim), dtype=np.float32)) * scale
    v = rng.standard_normal((n, kv_heads * head_dim), dtype=np.float32)
    got = kv.prefill_rows(q, k, v)
    want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
    # scores reach 9 * 64 * 0.64 / 8 = 46: on bf16 layers two 8-bit terms a query, 2^-17 of the score as an
    # error of the exponent; on f32 ones a rounding of 2^-24 of the score at each of 64 sums
    assert np.abs(got - want).max() <= 46 * np.abs(v).max() * (2.0 ** -16 if element == "bf16" else 64 * 2.0 ** -24)


def test_f32_chunk_is_no_less_exact_than_f32_sums(state, shape):
    """Three bf16 terms a factor, against 64 bits: no further off than torch's own f32 attention over
    the same rows, whose sums are f32 products (a margin of 1.5 for the order of the sums)."""
    import torch
    q_heads, kv_heads, head_dim, base, n = 8, 2, 128, 700, 96
    gen = torch.Generator().manual_seed(5)
    k, v = (torch.randn(base + n, kv_heads * head_dim, generator=gen) * torch.exp(torch.randn(base + n, 1, generator=gen)) for _ in range(2))
    q = torch.randn(n, q_heads * head_dim, generator=gen)
    kv = state.full_attention_f32(base + n, q_heads, kv_heads, head_dim)
    kv.seed(k[:base].numpy(), v[:base].numpy(), base)
    got = torch.from_numpy(kv.prefill_rows(q.numpy(), k[base:].numpy(), v[base:].numpy()))

    def attend(dt):
        out = torch.empty(n, q_heads * head_dim, dtype=dt)
        hidden = torch.arange(base + n)[None] > base + torch.arange(n)[:, None]
        for h in range(q_heads):
            g = h // (q_heads // kv_heads)
            cols, own = slice(h * head_dim, (h + 1) * head_dim), slice(g * head_dim, (g + 1) * head_dim)
            s = q[:, cols].to(dt) @ k[:, own].to(dt).T.contiguous() / head_dim ** 0.5
            out[:, cols] = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[:, own].to(dt)
        return out

    want, f32 = attend(torch.float64), attend(torch.float32)
    assert (got.double() - want).norm() <= 1.5 * (f32.double() - want).norm()


@pytest.mark.parametrize("head_dim,window,base,rows", [
    (72, 0, 2661, 509),     # padded head, a page that the cache and the chunk share, slots that do not fill a workgroup
    (128, 0, 2673, 512),    # the last group of eight pages cut after one
    (128, 3200, 3507, 500), # a ring: old pages, then pages of the chunk's own rows
])
def test_chunks_that_quarters_take(state, head_dim, window, base, rows):
    """208 workgroups of 64 slots over about 200 pages: four parts of two wavefronts with two tiles each."""
    import torch
    heads, n = 26, base + rows
    gen = torch.Generator().manual_seed(base)
    k, v = (torch.randn(n, heads * head_dim, generator=gen) for _ in range(2))
    q = torch.randn(rows, heads * head_dim, generator=gen)
    kv = state.full_attention_bf16(n, heads, heads, head_dim, window=window)
    kv.set_block_table(np.random.default_rng(base).permutation(kv.pages()).astype(np.int32))
    kv.seed(k[:base].numpy(), v[:base].numpy(), base)
    got = torch.from_numpy(kv.prefill_rows(q.numpy(), k[base:].numpy(), v[base:].numpy()))
    at, row = torch.arange(n)[None], base + torch.arange(rows)[:, None]
    hidden = (at > row) | (at <= row - window if window else at < 0)
    k, v = (x.bfloat16().double() for x in (k, v))
    want = torch.empty(rows, heads * head_dim, dtype=torch.float64)
    for h in range(heads):
        cols = slice(h * head_dim, (h + 1) * head_dim)
        s = q[:, cols].double() @ k[:, cols].T.contiguous() / head_dim ** 0.5
        want[:, cols] = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[:, cols]
    # queries and probabilities in two 8-bit terms: 2^-16 of scores up to 6, and of the probabilities
    assert (got.double() - want).abs().max() <= 7 * 2.0 ** -16 * want.abs().max()


@pytest.mark.parametrize("heads,head_dim,window,base,rows", [
    (26, 64, 0, 0, 512),     # 208 workgroups of 64 slots from an empty cache: the tile kernel
    (26, 64, 0, 0, 480),     # 208 too, but fewer pairs: the multi-query mode
    (27, 96, 0, 37, 481),    # 216, whose last ones are half full
    (32, 40, 1024, 0, 511),  # 256, on a ring that has not wrapped
])
@pytest.mark.parametrize("element", ["bf16", "f32"])
def test_first_chunks_of_a_workgroup_to_each_compute_unit(state, element, heads, head_dim, window, base, rows):
    """Short walks of as many slots as the compute units take at once, on both sides of the line between the kernels."""
    import torch
    n = base + rows
    gen = torch.Generator().manual_seed(n)
    k, v = (torch.randn(n, heads * head_dim, generator=gen) for _ in range(2))
    q = torch.randn(rows, heads * head_dim, generator=gen)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(n, heads, heads, head_dim, window=window)
    if base:
        kv.seed(k[:base].numpy(), v[:base].numpy(), base)
    got = torch.from_numpy(kv.prefill_rows(q.numpy(), k[base:].numpy(), v[base:].numpy()))
    hidden = torch.arange(n)[None] > base + torch.arange(rows)[:, None]
    k, v = (x.double() if element == "f32" else x.bfloat16().double() for x in (k, v))
    want = torch.empty(rows, heads * head_dim, dtype=torch.float64)
    for h in range(heads):
        cols = slice(h * head_dim, (h + 1) * head_dim)
        s = q[:, cols].double() @ k[:, cols].T.contiguous() / head_dim ** 0.5
        want[:, cols] = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[:, cols]
    # bf16: queries and probabilities in two 8-bit terms, 2^-16 of scores up to 6, and of the probabilities; f32: sums of up to 600 products
    assert (got.double() - want).abs().max() <= (2e-5 if element == "f32" else 7 * 2.0 ** -16 * want.abs().max())


@pytest.mark.parametrize("dims,base,rows", [((8, 2, 64), 1500, 70), ((28, 4, 128), 516, 448), ((12, 4, 96), 700, 200), ((16, 2, 256), 200, 300),
                                            ((8, 2, 512), 32, 256)])
def test_terms_of_queries_and_probabilities_are_rounded(state, shape, dims, base, rows):
    """Two bf16 terms each, rounded to nearest: 2^-18 relative at most in a probability and in a query element, whose effects on a
    context are of either sign. (A first term that is cut off doubles the largest error of a probability: 1.4 times 2^-18 in all.)"""
    import torch
    q_heads, kv_heads, head_dim = dims
    n = base + rows
    gen = torch.Generator().manual_seed(n)
    k, v = (torch.randn(n, kv_heads * head_dim, generator=gen) for _ in range(2))
    q = torch.randn(rows, q_heads * head_dim, generator=gen)
    kv = state.full_attention_bf16(n, q_heads, kv_heads, head_dim)
    kv.set_block_table(np.random.default_rng(base).permutation(kv.pages()).astype(np.int32))
    kv.seed(k[:base].numpy(), v[:base].numpy(), base)
    got = torch.from_numpy(kv.prefill_rows(q.numpy(), k[base:].numpy(), v[base:].numpy()))
    hidden = torch.arange(n)[None] > base + torch.arange(rows)[:, None]
    k, v = (x.bfloat16().double() for x in (k, v))
    want = torch.empty(rows, q_heads * head_dim, dtype=torch.float64)
    for h in range(q_heads):
        own, group = slice(h * head_dim, (h + 1) * head_dim), h // (q_heads // kv_heads)
        cols = slice(group * head_dim, (group + 1) * head_dim)
        s = q[:, own].double() @ k[:, cols].T.contiguous() / head_dim ** 0.5
        want[:, own] = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[:, cols]
    assert (got.double() - want).norm() <= 1.15 * 2.0 ** -18 * want.norm()


@pytest.mark.parametrize("dims,window,start,counts", [
    ((8, 2, 64), 0, 0, (2, 16, 15, 7, 16)),     # from an empty cache, across and up to page edges
    ((16, 2, 256), 0, 1021, (6, 16, 3, 16)),    # several query tiles, whose last one stores; rows in two splits' pages
    ((32, 8, 128), 0, 2300, (12, 2, 16)),
    ((20, 1, 128), 0, 40, (5, 1, 16)),          # more heads a group than a tile has slots
    ((3, 1, 18), 0, 30, (4, 16)),               # no 16-byte loads, padded head
    ((4, 2, 320), 0, 333, (16, 5)),             # several units a thread
    ((8, 2, 64), 10, 20, (9, 12)),              # a ring layer: appended by a launch of its own
])
def test_few_rows_are_appended_by_the_attention_launch(state, dims, window, start, counts):
    q_heads, kv_heads, head_dim = dims
    rng = np.random.default_rng(start + head_dim)
    kv = state.full_attention_bf16(start + sum(counts), q_heads, kv_heads, head_dim, window=window)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("bf16r")
    kv_dim = kv_heads * head_dim
    if start:
        k, v = (rng.standard_normal((start, kv_dim), dtype=np.float32) for _ in range(2))
        kv.seed(k, v, start)
        cache.append_batch(k, v, lay)
    for c in counts:
        q = rng.standard_normal((c, q_heads * head_dim), dtype=np.float32)
        k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
        got = kv.prefill_rows(q, k, v)
        want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
        assert np.abs(got - want).max() <= 1e-4, c
    first = max(0, kv.len() - window) if window else 0
    gk, gv = kv.read_rows_f32(first, kv.len() - first)
    assert np.array_equal(gk, cache.keys()[first:]) and np.array_equal(gv, cache.values()[first:])


@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
@pytest.mark.parametrize("dims,base,counts", [
    ((16, 2, 256), 700, (30, 31)),  # 15 and 16 tiles of 16 slots, three splits each
    ((16, 2, 256), 1500, (17, 31, 32)),  # 9 tiles in 14 splits, whose workgroups want a page on several XCDs; 16 in 8, on one
    ((64, 8, 32), 5, (64, 66)),     # 32 tiles a kv head, and more
    ((16, 2, 256), 5000, (6, 12)),  # 42 and 21 splits over two kv heads: taken in whole eights, 40 and 20
    ((6, 3, 48), 3100, (20, 130)),  # no power of two of kv heads
])
def test_rows_whose_tiles_share_pages(state, element, tol, dims, base, counts):
    q_heads, kv_heads, head_dim = dims
    rng = np.random.default_rng(base + head_dim)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(base + sum(counts), q_heads, kv_heads, head_dim)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    kv_dim = kv_heads * head_dim
    k, v = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
    kv.seed(k, v, base)
    cache.append_batch(k, v, lay)
    for c in counts:
        q = rng.standard_normal((c, q_heads * head_dim), dtype=np.float32)
        k, v = (rng.standard_normal((c, kv_dim), dtype=np.float32) for _ in range(2))
        got = kv.prefill_rows(q, k, v)
        want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
        assert np.abs(got - want).max() <= tol, c


@pytest.mark.parametrize("head_dim,window,base", [(64, 0, 61), (128, 0, 900), (256, 0, 61), (256, 0, 900), (40, 0, 900),
                                                  (64, 70, 61), (128, 900, 1200)])  # one split, several; rings
def test_infinite_rows_of_an_f32_chunk(state, shape, head_dim, window, base):
    """A live f32 row with an infinity gives what f32 products give, and only to the rows that attend it: an
    infinite V element that column of their contexts, an infinite K element weight zero or a NaN context as the
    query's sign there has it, an infinite query element its own head's context."""
    q_heads, kv_heads, rows = 4, 2, 150
    kv_dim, q_dim = kv_heads * head_dim, q_heads * head_dim
    rng = np.random.default_rng(head_dim + window)
    kv = state.full_attention_f32(base + rows, q_heads, kv_heads, head_dim, window=window)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    lay = oracle.layout(q_heads, kv_heads, head_dim, sliding_window=window)
    cache = oracle.LayerKvCache("f32")
    k0, v0 = (rng.standard_normal((base, kv_dim), dtype=np.float32) for _ in range(2))
    kv.seed(k0, v0, base)
    cache.append_batch(k0, v0, lay)
    q = rng.standard_normal((rows, q_dim), dtype=np.float32)
    k, v = (rng.standard_normal((rows, kv_dim), dtype=np.float32) for _ in range(2))
    v[20, 3], v[100, head_dim + 7] = np.inf, -np.inf
    v[60, 5] = np.float32(3.4e38)      # finite: its first term, rounded, is not
    k[40, 9], k[120, head_dim + 2] = np.inf, -np.inf
    q[:, 9] = -np.abs(q[:, 9])         # head 0 gives that key weight zero; head 1 by its own sign
    q[140, 2 * head_dim + 1] = np.inf
    got = kv.prefill_rows(q, k, v)
    with np.errstate(all="ignore"):
        want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
    assert not np.isfinite(want).all() and np.isfinite(want[:20]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert (np.abs(got - want)[ok] <= 2e-5 * np.maximum(np.abs(want[ok]), 1.0)).all()


def test_f32_scores_of_one_product_each(state, shape):
    """Factors just below a bf16 value or one, one product a score, scores of a thousand: no further off
    than the kernel of f32 products (a margin of 1.5 for the order of the sums). With the terms cut off instead of
    rounded, what the products leave out is largest for these, and several times the rounding of f32 ones."""
    q_heads, kv_heads, head_dim, base, n = 2, 1, 32, 500, 64
    rng = np.random.default_rng(8)
    k = np.zeros((base + n, head_dim), np.float32)
    k[:, 3] = 16 * (1.5 - np.where(rng.random(base + n) < 0.5, 0, rng.integers(0x81, 0xa0, base + n)) * 2.0 ** -23)
    # queries whose products with the kernel's scale, 1 / sqrt(head_dim) in base 2, lie there
    scale = np.float32(1) / np.sqrt(np.float32(head_dim)) * np.float32(1.4426950408889634)
    some = (rng.uniform(240, 250, 1 << 20)).astype(np.float32)
    low = (some * scale).view(np.uint32) & 0xffff
    q = np.zeros((n, q_heads * head_dim), np.float32)
    q[:, 3::head_dim] = some[(low >= 0xff60) & (low < 0xff80)][:n * q_heads].reshape(n, q_heads)
    v = rng.standard_normal((base + n, head_dim), dtype=np.float32)
    want = np.empty((n, q_heads * head_dim))
    for h in range(q_heads):
        cols = slice(h * head_dim, (h + 1) * head_dim)
        s = q[:, cols].astype(np.float64) @ k.astype(np.float64).T / np.sqrt(head_dim)
        s[np.arange(base + n)[None] > base + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want[:, cols] = p / p.sum(1, keepdims=True) @ v

    def run():
        kv = state.full_attention_f32(base + n, q_heads, kv_heads, head_dim)
        kv.seed(k[:base], v[:base], base)
        out = kv.prefill_rows(q, k[base:], v[base:])
        kv.close()
        return np.linalg.norm(out - want)
    terms = run()
    os.environ["SKV_PREFILL_TILES"] = "0"
    skv.flags.reload()
    assert terms <= 1.5 * run()


@pytest.mark.parametrize("element", ["bf16", "f32"])
def test_values_near_the_top_of_the_range(state, shape, element):
    """Weights are never above one, so a context of 300 rows of 5e35 does not pass through an infinity: also where
    scores rise by less than what moves the softmax base."""
    rng = np.random.default_rng(6)
    q_heads, kv_heads, head_dim, n = 8, 2, 64, 300
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(n, q_heads, kv_heads, head_dim)
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    q = np.ones((n, q_heads * head_dim), np.float32)
    k = np.repeat(np.linspace(0.0, 0.6, n, dtype=np.float32)[:, None], kv_heads * head_dim, 1)   # scores 0 to 4.8, 6.9 in base 2
    v = (5e35 * (1.0 + 0.1 * rng.random((n, kv_heads * head_dim)))).astype(np.float32)
    got = kv.prefill_rows(q, k, v)
    want = oracle.cached_attention_prefill_rows(q, k, v, cache, lay)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert (np.abs(got - want) <= (1e-4 if element == "bf16" else 2e-5) * want).all()


@pytest.mark.parametrize("element", ["bf16", "f32"])
def test_errors_against_64_bits(state, shape, element):
    """Normal rows: on bf16 layers no more than the two 8-bit terms of queries and of probabilities leave (2^-17 of
    each at most, of either sign), on f32 ones no more than the kernel of f32 products (a margin of 1.05: the
    sums are in another order)."""
    import torch
    q_heads, kv_heads, head_dim, base, n = 8, 2, 128, 1536, 96
    gen = torch.Generator().manual_seed(9)
    k, v = (torch.randn(base + n, kv_heads * head_dim, generator=gen) for _ in range(2))
    q = torch.randn(n, q_heads * head_dim, generator=gen)

    def run():
        kv = (state.full_attention_f32 if element == "f32" else state.full_attention_bf16)(base + n, q_heads, kv_heads, head_dim)
        kv.seed(k[:base].numpy(), v[:base].numpy(), base)
        return torch.from_numpy(kv.prefill_rows(q.numpy(), k[base:].numpy(), v[base:].numpy())).double()
    got = run()
    keys, values = (x.double() if element == "f32" else x.bfloat16().double() for x in (k, v))
    hidden = torch.arange(base + n)[None] > base + torch.arange(n)[:, None]
    want = torch.empty_like(got)
    for h in range(q_heads):
        g = h // (q_heads // kv_heads)
        cols, own = slice(h * head_dim, (h + 1) * head_dim), slice(g * head_dim, (g + 1) * head_dim)
        s = q[:, cols].double() @ keys[:, own].T.contiguous() / head_dim ** 0.5
        want[:, cols] = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ values[:, own]
    bound = 2.0 ** -17 * want.norm()
    if element == "f32":
        os.environ["SKV_PREFILL_TILES"] = "0"
        skv.flags.reload()
        bound = 1.05 * (run() - want).norm()
    assert (got - want).norm() <= bound
