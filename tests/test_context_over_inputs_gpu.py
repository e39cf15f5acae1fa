"""A context that lies over what its own launch reads: its queries (exactly, or shifted by a head), a step's new row, a chunk's rows, the
gate. Whatever the launch's shape, unsplit ones among them, it is what the same call on a layer of its own writes elsewhere."""
import contextlib
import os

import numpy as np
import pytest
import torch

import saragossa_amd as skv

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _env(**env):
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    skv.flags.reload()
    try:
        yield
    finally:
        for k, was in saved.items():
            os.environ.pop(k) if was is None else os.environ.__setitem__(k, was)
        skv.flags.reload()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _twins(state, dims, element, rows, extra, window=0):
    """Two layers of the same rows, and the queries and rows that come next, as floats on the device"""
    q_heads, kv_heads, head_dim = dims
    rng = np.random.default_rng(rows * 7 + extra)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    k, v = (rng.standard_normal((rows + extra, kv_heads * head_dim), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((extra, q_heads * head_dim), dtype=np.float32)
    layers = []
    for _ in range(2):
        kv = make(rows + extra, q_heads, kv_heads, head_dim, window=window)
        if rows:
            kv.seed(k[:rows], v[:rows], rows)
        layers.append(kv)
    return layers, [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k[rows:], v[rows:])]


def _placed(src, lead, room):
    """A buffer of `room` floats that holds src from `lead` floats on"""
    buf = torch.zeros(max(room, lead + src.numel()), device="cuda")
    buf[lead:lead + src.numel()] = src.reshape(-1)
    return buf


STEPS = [((32, 8, 128), "bf16"), ((8, 2, 64), "bf16"), ((24, 1, 128), "bf16"), ((8, 8, 80), "bf16"), ((4, 2, 512), "bf16"),
         ((32, 8, 128), "f32"), ((24, 1, 64), "f32"), ((4, 2, 512), "f32")]


@pytest.mark.parametrize("dims,element", STEPS)
@pytest.mark.parametrize("rows", [15, 100, 200, 700])
@pytest.mark.parametrize("over", ["q", "in place", "k", "v"])
@pytest.mark.parametrize("env", [{}, {"RETI_RUST_SDPA_2PASS": "0"}, {"RETI_RUST_FLASH_SDPA": "0"}], ids=["", "unsplit", "plain"])
def test_steps(state, dims, element, rows, over, env):
    with _env(**env):
        (one, other), (q, k, v) = _twins(state, dims, element, rows, 1)
        want = torch.zeros(q.numel(), device="cuda")
        other.encode_decode_step(_stream(), k.data_ptr(), 0, v.data_ptr(), 0, q.data_ptr(), want.data_ptr())
        lead = 0 if over == "in place" else dims[2]
        under = over if over in "kv" else "q"
        buf = {n: _placed(a, lead if n == under else 0, lead + q.numel()) for n, a in zip("qkv", (q, k, v))}
        at = {n: b.data_ptr() + (lead * 4 if n == under else 0) for n, b in buf.items()}
        one.encode_decode_step(_stream(), at["k"], 0, at["v"], 0, at["q"], buf[under].data_ptr())
        assert (buf[under][:q.numel()] - want).abs().max().item() <= 2e-5
        assert one.len() == rows + 1


@pytest.mark.parametrize("element", ["bf16", "f32"])
@pytest.mark.parametrize("dims", [(16, 2, 256), (4, 2, 512), (24, 1, 64)])
@pytest.mark.parametrize("rows", [20, 100, 900])
@pytest.mark.parametrize("lead", [0, 64])
@pytest.mark.parametrize("fused", ["1", "0"])
def test_gated_steps(state, dims, element, rows, lead, fused):
    """The context lies over the gated projection: the gate of a later head under that of an earlier one"""
    q_heads, kv_heads, head_dim = dims
    with _env(SKV_FUSED_APPEND=fused):
        (one, other), (q, k, v) = _twins(state, dims, element, rows, 1)
        qg = torch.randn(2 * q.numel(), device="cuda")
        rope = state.rope_table(rows + 1, 64, 10000.0)
        want = torch.zeros(q.numel(), device="cuda")
        other.encode_decode_step_gated(_stream(), rope, rows, qg.data_ptr(), 0, k.data_ptr(), 0, v.data_ptr(), 0, None, None, 1e-6, 64.0,
                                       want.data_ptr())
        buf = _placed(qg, lead, 0)
        one.encode_decode_step_gated(_stream(), rope, rows, buf.data_ptr(), lead * 4, k.data_ptr(), 0, v.data_ptr(), 0, None, None, 1e-6, 64.0,
                                     buf.data_ptr())
        assert (buf[:q.numel()] - want).abs().max().item() <= 2e-5


@pytest.mark.parametrize("dims,element", [((8, 2, 64), "bf16"), ((32, 8, 128), "bf16"), ((4, 2, 512), "bf16"), ((8, 2, 64), "f32")])
@pytest.mark.parametrize("lens", [[100, 20, 60], [100, 700, 40], [200, 300, 100], [900, 800, 700]])
@pytest.mark.parametrize("over", ["next query", "in place", "own query", "last rows"])
@pytest.mark.parametrize("twopass", ["1", "0"])
def test_batches(state, dims, element, lens, over, twopass):
    """A sequence's context over the next one's query, over its own, exactly or shifted by a head, or over rows of the last ones"""
    with _env(RETI_RUST_SDPA_2PASS=twopass):
        twins = [_twins(state, dims, element, rows, 1) for rows in lens]
        q, k, v = (torch.cat([t[1][i] for t in twins]) for i in range(3))
        n, q_dim, kv_dim = len(lens), q.shape[1], k.shape[1]
        want = torch.zeros(n, q_dim, device="cuda")
        rows = lambda t: [r.data_ptr() for r in t]
        skv.encode_decode_step_batch([t[0][1] for t in twins], _stream(), rows(k), rows(v), rows(q), rows(want))
        shift = {"next query": q_dim, "in place": 0, "own query": dims[2]}.get(over, 0)
        queries = torch.zeros((n + 1) * q_dim, device="cuda") # contexts `shift` floats behind the queries
        queries[:n * q_dim] = q.reshape(-1)
        keys = torch.zeros(n * max(q_dim, kv_dim), device="cuda")
        keys[:n * kv_dim] = k.reshape(-1)
        out = queries[shift:shift + n * q_dim] if over != "last rows" else keys[:n * q_dim]
        at = lambda t, d: [t.data_ptr() + i * d * 4 for i in range(n)]
        skv.encode_decode_step_batch([t[0][0] for t in twins], _stream(), at(keys, kv_dim), rows(v), at(queries, q_dim), at(out, q_dim))
        assert (out.reshape(n, q_dim) - want).abs().max().item() <= 2e-5


CHUNKS = [  # dims, element, rows in front, rows, window
    ((32, 8, 128), "bf16", 0, 512, 0),      # tile kernel, no split
    ((28, 4, 128), "bf16", 0, 700, 0),      # the same, more workgroups than the device holds
    ((32, 8, 128), "bf16", 0, 200, 0),      # multi-query mode
    ((8, 2, 64), "bf16", 60, 6, 0),         # few rows, appended by the launch
    ((8, 2, 64), "bf16", 3000, 12, 0),      # the same, split
    ((16, 8, 256), "bf16", 500, 512, 1024), # ring that has not wrapped
    ((32, 8, 128), "bf16", 600, 512, 512),  # ring that has, no split
    ((16, 8, 256), "bf16", 1100, 64, 1024), # ring that has, split
    ((8, 2, 512), "bf16", 30, 32, 0),
    ((32, 8, 128), "f32", 0, 512, 0),       # made terms
    ((32, 8, 128), "f32", 600, 512, 512),   # the same on a ring
    ((16, 2, 256), "f32", 0, 512, 0),       # made terms, heads above 128 dims
    ((16, 8, 256), "f32", 1100, 512, 1024), # the same on a ring
    ((32, 8, 128), "f32", 20, 20, 0),       # streaming
    ((8, 2, 512), "f32", 30, 64, 0),
    ((8, 2, 512), "f32", 300, 64, 256),     # two phases on a ring
]


@pytest.mark.parametrize("dims,element,rows,chunk,window,terms",
                         [c + (t,) for c in CHUNKS for t in (["1", "0"] if c[1] == "f32" else ["1"])])
@pytest.mark.parametrize("over", ["q", "in place", "k", "v"])
def test_chunks(state, dims, element, rows, chunk, window, over, terms):
    with _env(SKV_F32_TERMS=terms):
        (one, other), (q, k, v) = _twins(state, dims, element, rows, chunk, window)
        want = torch.zeros(q.numel(), device="cuda")
        other.encode_prefill_rows(_stream(), q.data_ptr(), k.data_ptr(), v.data_ptr(), chunk, want.data_ptr())
        lead = 0 if over == "in place" else 3 * dims[2]
        under = over if over in "kv" else "q"
        buf = {n: _placed(a, lead if n == under else 0, lead + q.numel()) for n, a in zip("qkv", (q, k, v))}
        at = {n: b.data_ptr() + (lead * 4 if n == under else 0) for n, b in buf.items()}
        one.encode_prefill_rows(_stream(), at["q"], at["k"], at["v"], chunk, buf[under].data_ptr())
        assert (buf[under][:q.numel()] - want).abs().max().item() <= 2e-5
        assert one.len() == rows + chunk


@pytest.mark.parametrize("terms", ["2", "0"])
def test_an_infinity_under_a_chunk_in_place(state, terms):
    """f32 heads above 128 dims: slots whose sums are not numbers are taken again from the queries, half of the columns at a time"""
    dims, chunk = (16, 2, 256), 512
    with _env(SKV_PREFILL_TILES="2", SKV_PREFILL_MAX_SPLITS="1", SKV_F32_TERMS=terms):
        (one, other), (q, k, v) = _twins(state, dims, "f32", 0, chunk)
        v[100, 5] = float("inf")
        want = torch.zeros_like(q)
        other.encode_prefill_rows(_stream(), q.data_ptr(), k.data_ptr(), v.data_ptr(), chunk, want.data_ptr())
        one.encode_prefill_rows(_stream(), q.data_ptr(), k.data_ptr(), v.data_ptr(), chunk, q.data_ptr())
        assert torch.isinf(want[100:, :8 * 256].reshape(-1, 8, 256)[:, :, 5]).all()
        finite = torch.isfinite(want)
        assert torch.equal(torch.isfinite(q), finite)
        assert (q[finite] - want[finite]).abs().max().item() <= 2e-5
